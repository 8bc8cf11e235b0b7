// Causal GQA prefill attention for gfx950: a bf16 MFMA path and an fp32 MFMA path.
//
// Algorithm (the reference's blocked causal GQA attention,
// src/deciax/kernels/attention/blocked.py:9-32, in the online form of its TPU
// flash kernel, src/deciax/kernels/attention/pallas.py:52-135): each
// workgroup owns one sequence, one KV head and a tile of query rows for all
// G = Hq / Hkv query heads sharing that KV head, so K/V tiles are staged in LDS
// once per group instead of being repeated per head (blocked.py:12-13 repeats
// them). Key tiles entirely outside the causal / sliding window are never
// visited; only tiles that straddle a boundary evaluate the mask.
//
// bf16 path, per wave (32 query rows of one head):
//   S^T = K Q^T  with 32x32x16 MFMAs: A = K rows from LDS, B = Q^T held in
//        registers for the whole key loop. Lane l then owns query (l % 32) and
//        16 keys per 32-key block, so row statistics are lane-local plus one
//        exchange with lane l ^ 32.
//   K rows are fed in the order kperm() so that the 8 keys a lane owns in
//   each half of a 32-key block are consecutive; those 8 scores become, after
//   bf16 rounding, the lane's B operand of O^T = V^T P^T directly, and the A
//   operand is one 16-byte read of the V^T tile (V transposed, [D][64] in LDS).
//
// Softmax: with logit soft-capping (Gemma-2, cap <= 56) every capped score
// lies in (-cap, cap), so p = exp(t - cap/2) is computed with a fixed shift:
// no running max, no rescaling of the O accumulator, no cross-lane max.
// t - cap/2 = cap/2 - 2 cap / (1 + e^{2x}), x = scale * s / cap, hence in log2
// units c3 + c2 / (1 + exp2(c1 s)) with c1 = 2 log2(e) scale / cap,
// c2 = -2 cap log2(e), c3 = cap log2(e) / 2. The kernel multiplies q by c1 as it
// loads it (one bf16 rounding of c1 q), so the MFMA yields c1 s directly, and
// folds c2 into the reciprocal:
//   p = exp2(c3 + 1 / fma(exp2(c1 s), 1/c2, 1/c2)),
// three transcendentals and two ordinary VALU operations per score.
// p stays within [e^{-3cap/2}, e^{cap/2}] — normal fp32 and bf16 numbers for
// cap <= 56 — and softmax is invariant to the shift. Without soft-capping (or
// for larger caps) the kernel keeps the usual running max in log2 units.
// P is rounded to bf16 before P.V (the reference rounds the normalised
// weights to q.dtype, blocked.py:27); O is divided by the fp32 row sum.
#include "common.h"
#include "kernels.h"

namespace {

constexpr int THREADS = 256;        // the V^T transpose and the mask words
constexpr int BKV = 64;     // V^T block alignment of dx_transpose_v
// bf16 path: waves per workgroup and LDS ring depth. The long form, 8 waves (two per SIMD, 32 query rows
// each) over a 4-stage ring (128 KB), runs one workgroup per CU. The short form, 4 waves over a 2-stage
// ring (64 KB), runs two workgroups per CU that fall out of step with each other, so one's prologue,
// epilogue and barrier waits overlap the other's key loop; it halves the query rows per staged K/V tile.
// Head_dim 128 takes the short form when a query row sees 2048 keys or fewer on average (window <= 2048,
// or causal sequences up to 4096): 27B heads, 8 x 2048 -4%, window 512 -12 to -15%, window 1024 -5 to -10%, 16 x 3400
// -2%; on longer spans it measured +0.2 to +1.1% (4 x 16384). Head_dim 64 takes it up to 4096 keys: its 32 KB ring puts
// three workgroups on a CU, and half the query rows spread small launches further (us of the kernel alone, 12 heads, no
// soft-cap, long -> short: 2 x 1021 37 -> 31, 4 x 2048 105 -> 79, 1 x 2048 49 -> 38, 8 x 1021 57 -> 47, 4 x 8192 causal
// 605 -> 554). Head_dim 256: the short form measured 6-11% slower. Where the long one has at most a workgroup per CU, four
// waves over the same 4-stage ring (one per SIMD) halve what the longest workgroup has to do: kernel alone, 16/8 heads,
// soft-capped, 1 x 736 40 -> 32 us, 1 x 2000 103 -> 87, 1 x 3300 162 -> 137 (208 workgroups of 8 waves), 4 x 1000 61 -> 58
// (256); 1 x 4500 (288) is even, 8 x 1000 (512) 84 -> 114. Two waves measured like four. All forms give the same bits.
// bf16 grid order switch (see attn_bf16_kernel). Whole units per XCD measured 3-9% faster at 3257-4096
// tokens (16 sequences, 9B and 27B heads), 2% slower at 8 x 3072 and 15% slower at 8 x 2048.
constexpr int SHORT_SEQ = 3072;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float NEG_BIG = -1e30f;  // the reference's MASK_FILL (reference.py:8)

// MODE_CAP: running max with a soft-cap (those beyond the fixed shift). A mode of its own: the sixteen tanhf of a
// block would otherwise sit in the loop of every launch without one.
enum { MODE_FIXED = 0, MODE_ONLINE = 1, MODE_CAP = 2 };

DX_DEVICE bool visible(int qi, int key, int len, int window, int causal) {
  if (key >= len) return false;
  if (causal) return key <= qi && (window <= 0 || key > qi - window);
  return window <= 0 || abs(qi - key) <= window;
}

// K tile in LDS: [TK keys][D], 16-byte chunk c of row r at slot c ^ k_swz<D>(r) (see below).

// V^T tile in LDS: [D][T keys]; with 64-byte rows (T = 32) chunk c of row r sits at slot c ^ ((r >> 2) & 3),
// with 128-byte rows (T = 64) at c ^ ((r >> 1) & 7): the 16 rows one fragment read touches per pass fill
// all 16 chunk slots of a 256-byte bank line.
template <int T>
DX_DEVICE int vt_swz(int row) {
  if constexpr (T == 32) return (row >> 2) & 3;
  else return (row >> 1) & 7;  // 128-byte rows
}
template <int T>
DX_DEVICE int vt_off(int row, int chunk) { return row * T + ((chunk ^ vt_swz<T>(row)) << 3); }

// MFMA row vk of a 32-key block reads key kperm(vk). The output register r of
// lane-half hh then holds key 16 (r >> 3) + 8 hh + (r & 7).
DX_DEVICE int kperm(int vk) { return 16 * (vk >> 4) + 8 * ((vk >> 2) & 1) + 4 * ((vk >> 3) & 1) + (vk & 3); }

// Direct-to-LDS loads: instruction j of a wave's share fills 1 KB of LDS (64 lanes x 16 bytes) at a
// wave-uniform base; each lane fetches the global chunk whose swizzled slot it fills.
typedef __attribute__((address_space(3))) void lds_void;

DX_DEVICE __amdgpu_buffer_rsrc_t make_rsrc(const uint16_t *base, long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, (int)bytes, 0x00020000);
}

// 16 bytes per lane from a buffer resource into LDS at lds + 16 * lane. The builtin is compiled in the
// device pass only: this clang drops a kernel's host-side symbols when the host pass sees it.
DX_DEVICE void lds_load16(__amdgpu_buffer_rsrc_t rsrc, uint16_t *lds, int voffset) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void *)lds, 16, voffset, 0, 0, 0);
#endif
}

// Schedule n (LDS read, MFMA) pairs with the reads LEAD ahead: enough to cover LDS latency, few
// enough that the operand registers in flight stay small.
template <int N>
DX_DEVICE void stream_sched() {
  constexpr int LEAD = 3;
  __builtin_amdgcn_sched_group_barrier(0x100, LEAD, 0);
#pragma unroll
  for (int t = 0; t < N - LEAD; ++t) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, LEAD, 0);
}

template <int D>
DX_DEVICE int k_swz(int row) {
  if constexpr (D / 8 >= 16) return row & 15;
  else return (row >> 1) & 7;
}

// bf16 path: WAVES waves (two per SIMD, the short or long form above), wave w = 32 query rows of head
// g * G + w % G. Each 64-key tile is processed in two 32-key halves (QK^T, softmax, PV per half) so a wave
// needs only 16 score registers and the other wave on its SIMD can run MFMAs while this one is in the
// softmax.
// Keys per tile: 32 at head_dim 256 (a 64-key tile would halve the ring depth), 64 below.
template <int D>
constexpr int tile_keys() { return D >= 256 ? 32 : 64; }

template <bool B>
struct Flag {
  static constexpr bool value = B;
};

// KM: a per-key mask (key_bits, key_words 32-bit words per sequence; bit j of word w of sequence b is key
// 32 w + j) hides keys beyond the causal / window rule. Tiles that hold a masked key take the masked body,
// and a query row that sees no key is written as zeros.
// Waves per SIMD that the registers are kept for: what the ring lets a CU hold. Head_dim 64's short form (32 KB) runs
// three: its loop waits on exponentials and LDS more than on the matrix core. Kernel alone, two -> three, us: 12 heads, 8 x
// 1021 58 -> 47, 4 x 2048 87 -> 79; 16 heads, 12 x 2048 284 -> 269, window 64 64 -> 53; four measured like three.
constexpr int waves_least(int d, int waves, int stages) {
  return waves * stages == 16 ? 1 : d == 64 && waves == 4 ? 3 : 2;
}
constexpr int waves_most(int d, int waves, int stages) { return d == 64 && waves == 4 && stages == 2 ? 3 : 2; }

template <int D, int G, int MODE, bool KM, int WAVES, int NSTAGE>
__global__ void __launch_bounds__(64 * WAVES)
__attribute__((amdgpu_waves_per_eu(waves_least(D, WAVES, NSTAGE), waves_most(D, WAVES, NSTAGE))))
attn_bf16_kernel(const uint16_t *__restrict__ Q, const uint16_t *__restrict__ K, const uint16_t *__restrict__ Vt,
                 uint16_t *__restrict__ O, const int32_t *__restrict__ seq_start,
                 const int32_t *__restrict__ seq_len, const int32_t *__restrict__ vt_start, long vt_seq_stride,
                 int max_seq_len, long q_stride, long k_stride, long vt_ld, long o_stride, float scale,
                 float softcap, int window, int causal, const uint32_t *__restrict__ key_bits, int key_words) {
  constexpr int TK = tile_keys<D>();
  constexpr int RG = WAVES / G;         // 32-row groups per head
  constexpr int BQ = 32 * RG;           // query rows per workgroup
  constexpr int KST = TK * D;           // elements of the K tile [TK][D]; the V^T tile [D][TK] follows
  constexpr int STAGE = 2 * TK * D;
  constexpr int NI = TK * D / 256;      // direct-to-LDS instructions per tile (K then V^T), 1 KB each
  constexpr int WI = NI / WAVES;        // per wave
  constexpr int NKS = D / 16;
  constexpr int NDB = D / 32;
  constexpr int CPR = D / 8;            // 16-byte chunks per K row
  static_assert(WI >= 2 && WI % 2 == 0 && NI % WAVES == 0, "tile too small for the wave count");
  static_assert(WAVES * 32 * D <= NSTAGE * STAGE, "the ring must hold every wave's 32 x D output tile");
  __shared__ __attribute__((aligned(1024))) uint16_t smem[NSTAGE * STAGE];

  // Grid order, the query tile index counted from the last (heaviest first):
  // - max_seq_len > SHORT_SEQ: (query tile, KV head, sequence), dealt out so that each XCD runs whole
  //   (sequence, KV head) units. Workgroups go to the 8 XCDs round-robin in dispatch order, each with its
  //   own L2, so dispatch p runs on XCD p % 8; unit u = 8 k + x takes XCD x's k-th run of query tiles.
  //   Every query tile of a unit reads the same K and V^T from key 0 (or the window start), so they hit
  //   in one L2 instead of being fetched once per XCD (9B batch: -7 to -9% per layer; 27B 4 x 16384:
  //   -6 to -14%). An XCD still walks its units in descriptor order, which the forward driver sorts
  //   longest first. Unit counts that are not a multiple of 8 keep the plain order.
  // - otherwise: (KV head, sequence, query tile), the heaviest tiles of every sequence first. With short
  //   sequences a single tile is a large share of a CU's work, so the order above leaves a tail
  //   (8 x 2048: 15% slower that way), while each (sequence, head)'s K and V^T fit in an XCD's L2.
  //   On ragged lengths up to 16K this order costs 25-35% instead: the concurrent streams scatter.
  const bool tile_major = max_seq_len <= SHORT_SEQ;
  int g, b, qt;
  if (tile_major) {
    g = blockIdx.x;
    b = blockIdx.y;
    qt = blockIdx.z;
  } else if ((gridDim.y * gridDim.z) % 8 == 0) {
    const long p = blockIdx.x + (long)gridDim.x * (blockIdx.y + (long)gridDim.y * blockIdx.z);
    const long idx = p >> 3, u = idx / gridDim.x * 8 + (p & 7);
    qt = (int)(idx % gridDim.x);
    g = (int)(u % gridDim.y);
    b = (int)(u / gridDim.y);
  } else {
    qt = blockIdx.x;
    g = blockIdx.y;
    b = blockIdx.z;
  }
  const int len = min(max(seq_len[b], 0), max_seq_len);
  const int ntiles = (max_seq_len + BQ - 1) / BQ;
  const int q0 = (ntiles - 1 - qt) * BQ;
  if (q0 >= len) return;
  const long start = seq_start[b];
  const long vts = vt_start ? (long)vt_start[b] : (long)b * vt_seq_stride;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int rg = wave / G, h = g * G + wave % G;
  const int qw0 = q0 + rg * 32, qw1 = qw0 + 31;
  const int qi = qw0 + lrow;

  bf16x8 qf[NKS];
  {
    const uint16_t *qp = Q + (start + min(qi, len - 1)) * q_stride + (long)h * D + lhalf * 8;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qf[ks] = as_bf16x8(*reinterpret_cast<const u32x4 *>(qp + ks * 16));
  }
  if constexpr (MODE == MODE_FIXED) {
    // q <- bf16(c1 q): the QK^T MFMAs then give the exponent c1 s of the fixed-shift softmax below
    const float c1 = 2.f * LOG2E * scale / softcap;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      u32x4 w = __builtin_bit_cast(u32x4, qf[ks]);
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = pack_bf2(lo_bf(w[i]) * c1, hi_bf(w[i]) * c1);
      qf[ks] = as_bf16x8(w);
    }
  }

  const int qlast = min(q0 + BQ, len) - 1;
  int klo, khi;
  if (causal) {
    khi = qlast + 1;
    klo = window > 0 ? max(0, q0 - window + 1) : 0;
  } else {
    khi = window > 0 ? min(len, qlast + window + 1) : len;
    klo = window > 0 ? max(0, q0 - window) : 0;
  }
  const int kt0 = klo / TK, kt1 = (khi + TK - 1) / TK;

  // K rows past len read as zero (outside the resource); V^T columns stay inside this sequence's
  // 64-aligned block, whose tail dx_transpose_v zero-fills. Each tile's resources are rebased at the
  // tile (scalar work), so the per-lane offsets below are loop-invariant.
  const uint16_t *kbase0 = K + start * k_stride + (long)g * D;
  const uint16_t *vbase0 = Vt + (long)g * D * vt_ld + vts;
  const long kbytes = (long)len * k_stride * 2;
  const long vbytes = ((long)(D - 1) * vt_ld + ((len + 63) & ~63)) * 2;
  // Wave w fills K instructions [w WI/2, (w + 1) WI/2) and as many V^T instructions. K instruction i
  // fills K slots [64 i, 64 i + 64): row p / CPR, chunk (p % CPR) ^ k_swz(row); V^T instruction i
  // fills row p / (TK / 8), chunk (p % (TK / 8)) ^ vt_swz(row).
  constexpr int WH = WI / 2;
  int koff[WH], voff[WH];
#pragma unroll
  for (int j = 0; j < WH; ++j) {
    const int p = (wave * WH + j) * 64 + lane;
    const int krow = p / CPR, kc = (p % CPR) ^ k_swz<D>(krow);
    koff[j] = (int)(krow * k_stride * 2) + kc * 16;
    const int vrow = p / (TK / 8), vc = (p % (TK / 8)) ^ vt_swz<TK>(vrow);
    voff[j] = (int)(vrow * vt_ld * 2) + vc * 16;
  }
  auto issue = [&](int kt, int st) {
    uint16_t *base = smem + st * STAGE;
    const long kb = (long)kt * TK;
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kbase0 + kb * k_stride, max(kbytes - kb * k_stride * 2, 0L));
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vbase0 + kb, vbytes - kb * 2);
#pragma unroll
    for (int j = 0; j < WH; ++j) {
      lds_load16(rk, base + (wave * WH + j) * 512, koff[j]);
      lds_load16(rv, base + KST + (wave * WH + j) * 512, voff[j]);
    }
  };

  floatx16 o[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float lsum = 0.f;
  float mrun = NEG_BIG;

  const float c2inv = 1.f / (-2.f * LOG2E * softcap);
  const float c3 = 0.5f * LOG2E * softcap;

  // Which 32-key blocks this wave's rows see: active = some key visible, masked = some key hidden.
  auto block_state = [&](const int kbase, bool &need_mask) {
    bool active = qw0 < len;
    need_mask = kbase + 32 > len;
    if (causal) {
      active = active && kbase <= qw1 && !(window > 0 && kbase + 31 <= qw0 - window);
      need_mask = need_mask || kbase + 31 > qw0 || (window > 0 && kbase <= qw1 - window);
    } else if (window > 0) {
      active = active && kbase <= qw1 + window && kbase + 31 >= qw0 - window;
      need_mask = need_mask || kbase < qw1 - window || kbase + 31 > qw0 + window;
    }
    return active;
  };
  // Visible keys of row qi form one interval [vlo, vhi].
  int vlo, vhi;
  if (causal) {
    vhi = min(qi, len - 1);
    vlo = window > 0 ? qi - window + 1 : 0;
  } else {
    vhi = window > 0 ? min(qi + window, len - 1) : len - 1;
    vlo = window > 0 ? qi - window : 0;
  }

  // One 32-key block kb of the tile in stage sk (K, then V^T at sk + KST): S^T = K Q^T, softmax,
  // O^T += V^T P^T. MASKED evaluates the causal / window / length mask and skips blocks no row sees.
  auto block = [&](const uint16_t *sk, const int kbase, const int kb, auto masked) {
    constexpr bool M = decltype(masked)::value;
    if constexpr (M) {
      bool need_mask;
      if (!block_state(kbase, need_mask)) return;
    }
    floatx16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
    {
      // for ks and ks + 8 the swizzled slots differ by the same 16 chunks: 8 lane offsets serve all 16
      const int krow = kb * 32 + kperm(lrow);
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const int lo = (((ks & 7) * 2 + lhalf) ^ k_swz<D>(krow)) << 3;
        s = mfma32(as_bf16x8(*reinterpret_cast<const u32x4 *>(sk + krow * D + (ks & ~7) * 16 + lo)), qf[ks], s);
      }
      stream_sched<NKS>();  // keep only a few K fragments live at once
    }
    // key of score r: kbase + 16 (r >> 3) + 8 lhalf + (r & 7); visible iff inside [vlo, vhi] (and, with a
    // key mask, its bit is set: kbase is a multiple of 32, so the block's 32 keys are one mask word)
    const int mlo = vlo - kbase - 8 * lhalf, mhi = vhi - kbase - 8 * lhalf;
    uint32_t kbits = 0xffffffffu;
    if constexpr (KM && M) kbits = key_bits[(long)b * key_words + (kbase >> 5)] >> (8 * lhalf);
    auto keep = [&](int r) {
      const int j = 16 * (r >> 3) + (r & 7);
      if constexpr (KM) return j >= mlo && j <= mhi && ((kbits >> j) & 1u);
      else return j >= mlo && j <= mhi;
    };
    if constexpr (MODE == MODE_FIXED) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float e = fast_exp2(s[r]);  // s[r] = c1 * score: q was scaled by c1 at load
        float p = fast_exp2(fast_rcp(__builtin_fmaf(e, c2inv, c2inv)) + c3);
        if constexpr (M) p = keep(r) ? p : 0.f;
        s[r] = p;
        lsum += p;
      }
    } else {
      // The maximum is raised once per 32-key block and P rounded against it, so outputs depend on that step (64 keys
      // under one maximum: 4 x 2048 172 us for 183, outputs moved by 1e-3 of their size). What rounds where is spelled
      // out, so that no change of the code around it moves them: interior blocks round the exponent once, in the fma,
      // masked ones after each operation, which changes a P in some 1e5 by its last bit.
#pragma clang fp contract(off)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] *= scale;
        if constexpr (MODE == MODE_CAP) s[r] = softcap * tanhf(s[r] / softcap);
      }
      float smax = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if constexpr (M) smax = keep(r) ? fmaxf(smax, s[r]) : smax;
        else smax = fmaxf(smax, s[r]);
      }
      const float tmax = fmaxf(smax * LOG2E, NEG_BIG);
      const float mnew = fmaxf(mrun, fmaxf(tmax, __shfl_xor(tmax, 32, 64)));
      const float alpha = fast_exp2(mrun - mnew);
      if (__builtin_amdgcn_ballot_w64(mnew != mrun)) {  // else alpha is 1 for all 32 rows
#pragma unroll
        for (int i = 0; i < NDB; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
      }
      mrun = mnew;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float p;
        if constexpr (M) p = keep(r) ? fast_exp2(s[r] * LOG2E - mnew) : 0.f;
        else p = fast_exp2(__builtin_fmaf(s[r], LOG2E, -mnew));
        s[r] = p;
        lsum = r == 0 ? __builtin_fmaf(lsum, alpha, p) : lsum + p;
      }
    }
    bf16x8 pf[2];
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      u32x4 w;
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = pack_bf2(s[8 * h2 + 2 * i], s[8 * h2 + 2 * i + 1]);
      pf[h2] = as_bf16x8(w);
    }
    const uint16_t *sv = sk + KST;
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      const int vrow = db * 32 + lrow;
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2)
        o[db] = mfma32(as_bf16x8(*reinterpret_cast<const u32x4 *>(sv + vt_off<TK>(vrow, kb * 4 + 2 * h2 + lhalf))),
                       pf[h2], o[db]);
    }
    stream_sched<2 * NDB>();
  };

  // Ring of NSTAGE tiles: tile kt sits in stage (kt - kt0) % NSTAGE, and tile kt + NSTAGE - 1 is
  // fetched while tile kt is multiplied (clamped: the last tiles reload themselves harmlessly).
  auto tile = [&](const int kt, auto masked) {
    issue(min(kt + NSTAGE - 1, kt1 - 1), (kt - kt0 + NSTAGE - 1) % NSTAGE);
    const uint16_t *sk = smem + ((kt - kt0) % NSTAGE) * STAGE;
#pragma unroll
    for (int kb = 0; kb < TK / 32; ++kb) block(sk, kt * TK + kb * 32, kb, masked);
    // tile kt + 1 has landed in every wave's share (the NSTAGE - 2 younger tiles may stay in flight)
    // and every wave is done reading tile kt, whose stage the next iteration refills. A plain s_barrier:
    // __syncthreads would also wait for the younger tiles' loads (its fence waits for all LDS writes).
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NSTAGE - 2) * WI) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  // Tiles [ta, tb) hold no key this wave's rows cannot see (all blocks active, none masked): they run
  // without any mask code. The tiles before and after take the masked body. Every wave runs one
  // iteration (one barrier) per tile, whichever body.
  int ta = kt1, tb = kt1;
  if (qw1 < len) {
    int lo_u = 0, hi_u = len - 32;  // first / last kbase of an unmasked block
    if (causal) {
      hi_u = min(hi_u, qw0 - 31);
      if (window > 0) lo_u = qw1 - window + 1;
    } else if (window > 0) {
      lo_u = qw1 - window;
      hi_u = min(hi_u, qw0 + window - 31);
    }
    lo_u = max(lo_u, 0);
    const int a = max(kt0, (lo_u + TK - 1) / TK);
    const int last = hi_u - (TK - 32);  // kbase of the tile's first block
    const int b = last < 0 ? kt0 : min(kt1, last / TK + 1);
    if (a < b) {
      ta = a;
      tb = b;
    }
  }

#pragma unroll
  for (int i = 0; i < NSTAGE - 1; ++i) issue(min(kt0 + i, kt1 - 1), i);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NSTAGE - 2) * WI) : "memory");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (KM) {
    // A tile of [ta, tb) whose keys the mask keeps entirely takes the unmasked body as well. Its mask
    // words are requested one tile ahead (scalar loads, which the tile's barrier wait covers).
    const uint32_t *const kw = key_bits + (long)b * key_words;
    auto full = [&](int kt) {
      bool f = true;
#pragma unroll
      for (int i = 0; i < TK / 32; ++i) f = f && kw[kt * (TK / 32) + i] == 0xffffffffu;
      return f;
    };
    for (int kt = kt0; kt < kt1; ++kt) {
      if (kt >= ta && kt < tb && full(kt)) {
        // a run of interior tiles whose keys the mask keeps, each next tile's words read before this one
        for (bool more = true; more; ++kt) {
          more = kt + 1 < tb && full(kt + 1);
          tile(kt, Flag<false>());
        }
        if (kt == kt1) break;
      }
      tile(kt, Flag<true>());
    }
  } else {
    for (int kt = kt0; kt < kt1; ++kt) {
      if (kt == ta) {
        for (; kt < tb; ++kt) tile(kt, Flag<false>());
        if (kt == kt1) break;
      }
      tile(kt, Flag<true>());
    }
  }
  // Every wave's ring loads have landed and no wave reads the ring any more: it now stages the output.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // Each lane holds 4-value pieces of its row qi scattered over the head's D columns; stored directly,
  // every store instruction would touch 32 rows (32 cache lines, 8 bytes each). The wave writes its
  // 32 x D bf16 tile to its own LDS region (row r's 16-byte chunk c at slot c ^ (r % CPR)), then each
  // store instruction writes whole contiguous rows, 16 bytes per lane.
  lsum += __shfl_xor(lsum, 32, 64);
  float inv = 1.f / lsum;
  if constexpr (KM) inv = lsum > 0.f ? inv : 0.f;
  // Lane indices derived anew here, through an opaque copy: values shared with the prologue would stay
  // live across the key loop, and the loop's schedule then keeps fewer fragment reads in flight.
  int el = (int)threadIdx.x & 63;
  asm volatile("" : "+v"(el));
  const int erow = el & 31, ehalf = el >> 5;
  uint16_t *stage = smem + wave * 32 * D;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int grp = 0; grp < 4; ++grp) {
      u32x2 w;
      w[0] = pack_bf2(o[db][grp * 4 + 0] * inv, o[db][grp * 4 + 1] * inv);
      w[1] = pack_bf2(o[db][grp * 4 + 2] * inv, o[db][grp * 4 + 3] * inv);
      const int chunk = db * 4 + grp;  // 16-byte chunk of the row; this lane fills its half ehalf
      *reinterpret_cast<u32x2 *>(stage + erow * D + ((chunk ^ (erow % CPR)) << 3) + ehalf * 4) = w;
    }
  __syncthreads();
  constexpr int RPI = 64 / CPR;  // rows per store instruction
#pragma unroll
  for (int i = 0; i < 32 / RPI; ++i) {
    const int r = i * RPI + el / CPR, c = el % CPR;
    if (qw0 + r < len)
      *reinterpret_cast<u32x4 *>(O + (start + qw0 + r) * o_stride + (long)h * D + c * 8) =
          *reinterpret_cast<const u32x4 *>(stage + r * D + ((c ^ (r % CPR)) << 3));
  }
}

// fp32 path, on the matrix core: v_mfma_f32_16x16x4_f32 (fp32 products and sums). A workgroup takes
// 16 QB query rows of one head; its WAVES waves take blocks of 16 SUB keys in turn, each with its own running max,
// row sum and O, merged through LDS at the end, so no barrier runs in the key loop. Operands go from global memory
// straight to MFMA lanes (the query tile, which every wave reads, through LDS). With r = lane % 16, g = lane / 16:
//   S^T = K Q^T    the four contraction indices of MFMA 4 c + e are dims 16 c + 4 g + e, so a lane reads 16 bytes
//                  of key row r per chunk c and a load covers 64 bytes of 16 rows. It gets back query r, keys
//                  4 g + 0..3. D / 32 partial sums per score: no MFMA waits for the one before, and 32 roundings
//                  in a row instead of D (error against 64 bits 1.9e-7, one chain 4.3e-7).
//   O^T += V^T P^T MFMA t contracts keys 4 g + t, whose probabilities the lane holds; output block 4 a + e is dims
//                  64 a + 4 r + e, so a load covers 256 bytes of 4 rows, and the lane ends up with the 16
//                  consecutive dims 64 a + 16 g + .. of query r.
// K of the next block is requested when this block's scores are done, V at the start of its block: each has half a
// block of MFMAs to land. What bounds it: the MFMAs and, at QB = 1 and head_dim 256, the 32 bytes per cycle and CU
// that K and V take from L2 (QB = 2 halves them).
// Measured, before (VALU kernel at head_dim 256, LDS-staged 32x32x2 MFMAs below it; us) -> now:
//   head_dim 256: 2 x 701, 8/4 heads, soft-capped 575 -> 82    4 x 1024, 32/8 heads 7890 -> 948 (73 TFLOP/s)
//   head_dim 128: 2 x 701, soft-capped 75 -> 43                4 x 1024, 32/8 heads 901 -> 454
//   head_dim 64:  2 x 701, soft-capped 45 -> 36                4 x 1024, 32/8 heads 550 -> 223
// with soft-capping the error at head_dim 64 and 128 fell from 2.0e-6 to 1.9e-7 (tanhf for the rcp / exp2 form).
DX_DEVICE floatx4 mfma16_f32(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Registers for two workgroups a CU at head_dim 64 (4 x 1024, 32/8 heads 275 -> 219 us), one above.
template <int D, int QB, int WAVES, int SUB>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : 1, D == 64 ? 4 : 1)))
attn_f32_kernel(const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V,
                    float *__restrict__ O, const int32_t *__restrict__ seq_start, const int32_t *__restrict__ seq_len,
                    int max_seq_len, int hq, int hkv, long q_stride, long k_stride, long v_stride, long o_stride,
                    float scale, float softcap, int window, int causal, const uint8_t *__restrict__ key_mask) {
  constexpr int C = D / 16, A = D / 64, KB = 16 * SUB, BQ = 16 * QB, OP = D + 4;
  constexpr int NC = D / 32;  // partial sums per score
  static_assert(D % 64 == 0 && KB <= 64 && (WAVES & (WAVES - 1)) == 0, "tile shape");
  __shared__ __attribute__((aligned(16))) float os[WAVES * BQ * OP];
  __shared__ float ms[WAVES][BQ], ls[WAVES][BQ];

  const int b = blockIdx.y, h = blockIdx.x % hq, g_kv = h / (hq / hkv);
  const int len = seq_len ? min(max(seq_len[b], 0), max_seq_len) : max_seq_len;  // null: a padded batch
  const int ntiles = (max_seq_len + BQ - 1) / BQ;
  const int q0 = (ntiles - 1 - (int)blockIdx.x / hq) * BQ;  // heaviest (last) query tiles first
  if (q0 >= len) return;
  const long start = seq_start ? (long)seq_start[b] : (long)b * max_seq_len;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;

  const int qlast = min(q0 + BQ, len) - 1;
  int klo, khi;
  if (causal) {
    khi = qlast + 1;
    klo = window > 0 ? max(0, q0 - window + 1) : 0;
  } else {
    khi = window > 0 ? min(len, qlast + window + 1) : len;
    klo = window > 0 ? max(0, q0 - window) : 0;
  }
  const float *const kp = K + start * k_stride + (long)g_kv * D + 4 * g;
  const float *const vp = V + start * v_stride + (long)g_kv * D + 4 * r;

  // the query tile, in the space that takes the waves' O later
  for (int idx = tid; idx < BQ * (D / 4); idx += 64 * WAVES) {
    const int q = idx / (D / 4), d = idx % (D / 4) * 4;
    *reinterpret_cast<floatx4 *>(os + q * OP + d) =
        *reinterpret_cast<const floatx4 *>(Q + (start + min(q0 + q, len - 1)) * q_stride + (long)h * D + d);
  }
  __syncthreads();
  const float *const qs = os + r * OP + 4 * g;
  floatx4 kf[SUB][C];
  auto load_k = [&](int k0) __attribute__((always_inline)) {  // rows past the sequence read its last one (masked)
#pragma unroll
    for (int s = 0; s < SUB; ++s) {
      const float *p = kp + (long)min(k0 + 16 * s + r, len - 1) * k_stride;
#pragma unroll
      for (int c = 0; c < C; ++c) kf[s][c] = *reinterpret_cast<const floatx4 *>(p + 16 * c);
    }
  };
  floatx4 o[QB][C];
  float m[QB], l[QB];
#pragma unroll
  for (int u = 0; u < QB; ++u) {
    m[u] = NEG_BIG;
    l[u] = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) o[u][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  // key block j goes to wave j % WAVES, counted from key 0: a row's sums then do not depend on the tile it is in, whose
  // height follows the size of the launch
  const int first = klo / KB;
  int k0 = (first + ((wave - first) & (WAVES - 1))) * KB;
  if (k0 < khi) load_k(k0);
  for (; k0 < khi; k0 += WAVES * KB) {
    floatx4 vf[SUB][4][A];
    // one mask byte per lane covers the block; bit 16 s + 4 g + t is the lane's key (s, t)
    const uint8_t mk = key_mask ? key_mask[start + min(k0 + min(lane, KB - 1), len - 1)] : (uint8_t)1;
#pragma unroll
    for (int s = 0; s < SUB; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float *p = vp + (long)min(k0 + 16 * s + 4 * g + t, len - 1) * v_stride;
#pragma unroll
        for (int a = 0; a < A; ++a) vf[s][t][a] = *reinterpret_cast<const floatx4 *>(p + 64 * a);
      }
    __builtin_amdgcn_sched_barrier(0);  // V's loads go out before the products
    floatx4 part[QB][SUB][NC];
#pragma unroll
    for (int u = 0; u < QB; ++u)
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int n = 0; n < NC; ++n) part[u][s][n] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < C; ++c) {
      floatx4 qf[QB];
#pragma unroll
      for (int u = 0; u < QB; ++u) qf[u] = *reinterpret_cast<const floatx4 *>(qs + 16 * u * OP + 16 * c);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int s = 0; s < SUB; ++s)
#pragma unroll
          for (int u = 0; u < QB; ++u) {
            floatx4 &acc = part[u][s][(4 * c + e) % NC];
            acc = mfma16_f32(kf[s][c][e], qf[u][e], acc);
          }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_k(k0 + WAVES * KB);
    floatx4 sc[QB][SUB];
#pragma unroll
    for (int u = 0; u < QB; ++u)
#pragma unroll
      for (int s = 0; s < SUB; ++s) {
#pragma unroll
        for (int w = NC / 2; w >= 1; w /= 2)
#pragma unroll
          for (int n = 0; n < w; ++n) part[u][s][n] += part[u][s][n + w];
        sc[u][s] = part[u][s][0];
      }
    const uint64_t bits = __builtin_amdgcn_ballot_w64(mk != 0) >> (4 * g);
#pragma unroll
    for (int u = 0; u < QB; ++u) {
      const int qi = q0 + 16 * u + r;
      if (softcap > 0.f) {
#pragma unroll
        for (int s = 0; s < SUB; ++s)
#pragma unroll
          for (int t = 0; t < 4; ++t) sc[u][s][t] = softcap * tanhf(sc[u][s][t] * scale / softcap);
      } else {
#pragma unroll
        for (int s = 0; s < SUB; ++s) sc[u][s] *= scale;
      }
      uint32_t vis = 0;
      float mx = NEG_BIG;
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const bool v = visible(qi, k0 + 16 * s + 4 * g + t, len, window, causal) && ((bits >> (16 * s + t)) & 1u);
          vis |= (uint32_t)v << (4 * s + t);
          mx = v ? fmaxf(mx, sc[u][s][t]) : mx;
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m[u], mx);
      const float alpha = expf(m[u] - mn);
      m[u] = mn;
      l[u] *= alpha;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {  // some row's running max moved
#pragma unroll
        for (int c = 0; c < C; ++c) o[u][c] *= alpha;
      }
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float p = ((vis >> (4 * s + t)) & 1u) ? expf(sc[u][s][t] - mn) : 0.f;
          sc[u][s][t] = p;
          l[u] += p;
        }
    }
    if (k0 + KB > len) {  // rows past the sequence count as zeros (their weight is 0, the last row's value may be infinite)
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (k0 + 16 * s + 4 * g + t >= len) {
#pragma unroll
            for (int a = 0; a < A; ++a) vf[s][t][a] = floatx4{0.f, 0.f, 0.f, 0.f};
          }
    }
#pragma unroll
    for (int s = 0; s < SUB; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int u = 0; u < QB; ++u) o[u][4 * a + e] = mfma16_f32(vf[s][t][a][e], sc[u][s][t], o[u][4 * a + e]);
  }
#pragma unroll
  for (int u = 0; u < QB; ++u) {
    l[u] += __shfl_xor(l[u], 16, 64);
    l[u] += __shfl_xor(l[u], 32, 64);
    if (u == 0) __syncthreads();  // the query tile is no longer read
    if (g == 0) {
      ms[wave][16 * u + r] = m[u];
      ls[wave][16 * u + r] = l[u];
    }
    float *row = os + (wave * BQ + 16 * u + r) * OP + 16 * g;
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<floatx4 *>(row + 64 * a + 4 * i) =
            floatx4{o[u][4 * a][i], o[u][4 * a + 1][i], o[u][4 * a + 2][i], o[u][4 * a + 3][i]};
  }
  __syncthreads();
  for (int idx = tid; idx < BQ * (D / 4); idx += 64 * WAVES) {
    const int q = idx / (D / 4), d = idx % (D / 4) * 4;
    if (q0 + q >= len) continue;
    float mx = ms[0][q];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) mx = fmaxf(mx, ms[w][q]);
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = expf(ms[w][q] - mx);
      acc += *reinterpret_cast<const floatx4 *>(os + (w * BQ + q) * OP + d) * f;
      sum += ls[w][q] * f;
    }
    floatx4 v = {0.f, 0.f, 0.f, 0.f};  // a row that sees no key: zeros
    if (sum > 0.f) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[e] / sum;
    }
    *reinterpret_cast<floatx4 *>(O + (start + q0 + q) * o_stride + (long)h * D + d) = v;
  }
}

// What one launch prepares for a padded batch (every sequence max_seq_len rows, back to back) beside the transpose:
// the sequence descriptors and the mask words. Null key_mask: a packed batch, descriptors given.
struct PaddedPrep {
  const uint8_t *key_mask = nullptr;
  uint32_t *bits = nullptr;
  int32_t *seq_start = nullptr, *seq_len = nullptr;
  int words = 0;
};

// V rows -> V^T tiles. Grid: (64-row tiles of the longest sequence, sequences,
// kv heads x D/64; with a PaddedPrep one more, whose workgroup x packs the 64 keys of tile x). Rows past seq_len up
// to the next multiple of 64 are written as zeros, so P.V never multiplies a zero probability by stale data.
template <bool PADDED>
__global__ void __launch_bounds__(THREADS)
transpose_v_kernel(const uint16_t *__restrict__ V, uint16_t *__restrict__ Vt, const int32_t *__restrict__ seq_start,
                   const int32_t *__restrict__ seq_len, const int32_t *__restrict__ vt_start, long vt_seq_stride,
                   int max_seq_len, int d, long v_stride, long vt_ld, PaddedPrep pp) {
  if constexpr (PADDED) {
    if (blockIdx.z == gridDim.z - 1) {
      const int b = blockIdx.y, key = (int)blockIdx.x * 64 + (int)threadIdx.x;
      if (threadIdx.x >= 64) return;
      const uint64_t m = __builtin_amdgcn_ballot_w64(key < max_seq_len && pp.key_mask[(long)b * max_seq_len + min(key, max_seq_len - 1)] != 0);
      if (threadIdx.x == 0) {
        uint32_t *w = pp.bits + (long)b * pp.words + 2 * blockIdx.x;
        w[0] = (uint32_t)m;
        w[1] = (uint32_t)(m >> 32);
        if (blockIdx.x == 0) {
          pp.seq_start[b] = b * max_seq_len;
          pp.seq_len[b] = max_seq_len;
        }
      }
      return;
    }
  }
  __shared__ uint16_t tile[64][66];
  const int b = blockIdx.y;
  const int len = PADDED ? max_seq_len : min(max(seq_len[b], 0), max_seq_len);
  const int p0 = blockIdx.x * 64;
  if (p0 >= len) return;
  const int dblocks = d / 64;
  const int g = blockIdx.z / dblocks, d0 = (blockIdx.z % dblocks) * 64;
  const long start = PADDED ? (long)b * max_seq_len : seq_start[b];
  const long vts = vt_start ? (long)vt_start[b] : (long)b * vt_seq_stride;
  const int tid = threadIdx.x;
  {
    const int row = tid >> 2, c = (tid & 3) * 16;
    u32x4 a = {0, 0, 0, 0}, bb = {0, 0, 0, 0};
    if (p0 + row < len) {
      const uint16_t *src = V + (start + p0 + row) * v_stride + (long)g * d + d0 + c;
      a = *reinterpret_cast<const u32x4 *>(src);
      bb = *reinterpret_cast<const u32x4 *>(src + 8);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      tile[row][c + 2 * i] = (uint16_t)(a[i] & 0xffff);
      tile[row][c + 2 * i + 1] = (uint16_t)(a[i] >> 16);
      tile[row][c + 8 + 2 * i] = (uint16_t)(bb[i] & 0xffff);
      tile[row][c + 8 + 2 * i + 1] = (uint16_t)(bb[i] >> 16);
    }
  }
  __syncthreads();
  {
    const int dr = tid >> 2, c = (tid & 3) * 16;
    u32x4 a, bb;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a[i] = (uint32_t)tile[c + 2 * i][dr] | ((uint32_t)tile[c + 2 * i + 1][dr] << 16);
      bb[i] = (uint32_t)tile[c + 8 + 2 * i][dr] | ((uint32_t)tile[c + 8 + 2 * i + 1][dr] << 16);
    }
    uint16_t *dst = Vt + ((long)g * d + d0 + dr) * vt_ld + vts + p0 + c;
    *reinterpret_cast<u32x4 *>(dst) = a;
    *reinterpret_cast<u32x4 *>(dst + 8) = bb;
  }
}

// Block (s, y): V^T rows [4 y, 4 y + 4) of sequence s, columns [seq_len, seq_len rounded up to 64) <- 0.
__global__ void __launch_bounds__(THREADS)
vt_zero_tails_kernel(uint16_t *__restrict__ Vt, const int32_t *__restrict__ seq_len,
                     const int32_t *__restrict__ vt_start, int vt_rows, long vt_ld) {
  const int len = max(seq_len[blockIdx.x], 0);
  const int row = blockIdx.y * (THREADS / 64) + (int)threadIdx.x / 64, j = len + (int)threadIdx.x % 64;
  if (row < vt_rows && j < ((len + 63) & ~63)) Vt[(long)row * vt_ld + vt_start[blockIdx.x] + j] = 0;
}

inline bool fixed_shift(const AttnArgs &a) { return a.softcap > 0.f && a.softcap <= 56.f; }

template <int D, int G, int W, int NS>
hipError_t launch_bf16_dgw(const AttnArgs &a, hipStream_t s) {
  constexpr int BQ = 32 * (W / G);
  const unsigned ntiles = (a.max_seq_len + BQ - 1) / BQ;
  const dim3 grid = a.max_seq_len <= SHORT_SEQ ? dim3(a.hkv, a.num_seqs, ntiles) : dim3(ntiles, a.hkv, a.num_seqs);
  auto kern = a.key_bits ? (fixed_shift(a) ? attn_bf16_kernel<D, G, MODE_FIXED, true, W, NS>
                                           : attn_bf16_kernel<D, G, MODE_ONLINE, true, W, NS>)
                         : (fixed_shift(a) ? attn_bf16_kernel<D, G, MODE_FIXED, false, W, NS>
                                           : attn_bf16_kernel<D, G, MODE_ONLINE, false, W, NS>);
  if constexpr (W == 8 || D == 128)
    if (a.softcap > 0.f && !fixed_shift(a))
      kern = a.key_bits ? attn_bf16_kernel<D, G, MODE_CAP, true, W, NS> : attn_bf16_kernel<D, G, MODE_CAP, false, W, NS>;
  kern<<<grid, dim3(64 * W), 0, s>>>(
      static_cast<const uint16_t *>(a.q), static_cast<const uint16_t *>(a.k), static_cast<const uint16_t *>(a.v),
      static_cast<uint16_t *>(a.out), a.seq_start, a.seq_len, a.vt_start, a.vt_seq_stride, a.max_seq_len,
      a.q_stride, a.k_stride, a.v_stride, a.out_stride, a.scale, a.softcap, a.window, a.causal, a.key_bits,
      a.key_words);
  return hipGetLastError();
}

// Keys a query row sees on average: the window, or half the longest sequence when causal and unwindowed.
inline long mean_key_span(const AttnArgs &a) {
  const long n = a.max_seq_len;
  const long w = a.window;
  if (a.causal) return w > 0 ? (w < n ? w : n) : n / 2;
  return w > 0 ? (2 * w < n ? 2 * w : n) : n;
}

template <int D, int G>
hipError_t launch_bf16_dg(const AttnArgs &a, hipStream_t s) {
  // MODE_CAP is built for the long form and the short one at head_dim 128
  if (D != 128 && a.softcap > 0.f && !fixed_shift(a)) return launch_bf16_dgw<D, G, 8, 4>(a, s);
  if constexpr (D <= 128)
    if (mean_key_span(a) <= (D == 64 ? 4096 : 2048)) return launch_bf16_dgw<D, G, 4, 2>(a, s);
  if constexpr (D == 256) {
    const long rows = 32 * (8 / G), long_form = (a.max_seq_len + rows - 1) / rows * a.hkv * a.num_seqs;
    if (long_form <= 256) return launch_bf16_dgw<D, G, 4, 4>(a, s);
  }
  return launch_bf16_dgw<D, G, 8, 4>(a, s);
}

template <int D>
hipError_t launch_bf16_d(const AttnArgs &a, hipStream_t s) {
  switch (a.hq / a.hkv) {
    case 1: return launch_bf16_dg<D, 1>(a, s);
    case 2: return launch_bf16_dg<D, 2>(a, s);
    case 4: return launch_bf16_dg<D, 4>(a, s);
  }
  return hipErrorInvalidValue;
}

template <int D, int QB, int W>
hipError_t launch_f32_dqw(const AttnArgs &a, hipStream_t s) {
  const dim3 grid((unsigned)((a.max_seq_len + 16 * QB - 1) / (16 * QB)) * a.hq, a.num_seqs);
  attn_f32_kernel<D, QB, W, 1><<<grid, dim3(64 * W), 0, s>>>(
      static_cast<const float *>(a.q), static_cast<const float *>(a.k), static_cast<const float *>(a.v),
      static_cast<float *>(a.out), a.seq_start, a.seq_len, a.max_seq_len, a.hq, a.hkv, a.q_stride, a.k_stride,
      a.v_stride, a.out_stride, a.scale, a.softcap, a.window, a.causal, a.key_mask);
  return hipGetLastError();
}

// Head_dim 64 and 128: 32 queries, 8 waves (two per SIMD; 4 waves, or 32 keys a step, measured 10 to 60% slower).
// Head_dim 256 has registers for 4 waves: 32 queries where that fills the CUs (4 x 1000, 8 heads 412 against 463 us),
// else 16 (1 x 97, 8 heads 17 against 22 us; 2 x 200, 4 heads 20 against 30).
template <int D>
hipError_t launch_f32_d(const AttnArgs &a, hipStream_t s) {
  if constexpr (D < 256) {
    return launch_f32_dqw<D, 2, 8>(a, s);
  } else {
    const long tiles = (long)((a.max_seq_len + 31) / 32) * a.hq * a.num_seqs;
    return tiles >= 256 ? launch_f32_dqw<D, 2, 4>(a, s) : launch_f32_dqw<D, 1, 4>(a, s);
  }
}

DX_DEVICE void widen(floatx4 v, float (&f)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) f[e] = v[e];
}
DX_DEVICE void widen(u32x4 v, float (&f)[8]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[2 * e] = lo_bf(v[e]);
    f[2 * e + 1] = hi_bf(v[e]);
  }
}
DX_DEVICE floatx4 narrow(const float (&f)[4]) { return floatx4{f[0], f[1], f[2], f[3]}; }
DX_DEVICE u32x4 narrow(const float (&f)[8]) {
  return u32x4{pack_bf2(f[0], f[1]), pack_bf2(f[2], f[3]), pack_bf2(f[4], f[5]), pack_bf2(f[6], f[7])};
}

// Padded batch: query rows that see no key get the mean of the sequence's num_k value rows (softmax of equal
// scores). A workgroup looks at 64 rows and one KV head. Row i sees keys [lo(i), hi(i)), and hi grows by one a row at
// most: the last kept key below hi(first row), found by all threads, and the 64 mask bytes from there on tell for each
// row whether its last kept key reaches lo(i). Almost every workgroup ends there. The others read the head's values, a
// 16-byte chunk (CHUNK: its type, VEC elements) of every SLICES-th key per thread, and add the threads' sums in LDS. The
// call at 4 x 2048, 32/8 heads x 128, with a full mask / one empty row / left padding: 207 / 244 / 223 us (192 / 611 / 593
// with all heads in one workgroup, one thread a column, and 64 keys under one maximum in the attention).
template <typename CHUNK, int VEC, int D>
__global__ void __launch_bounds__(THREADS)
fill_unseen_kernel(const CHUNK *__restrict__ V, CHUNK *__restrict__ O, const uint8_t *__restrict__ key_mask, int len,
                   int num_q, int num_k, int hq, int hkv, long v_stride, long o_stride, int window, int causal) {
  constexpr int CH = D / VEC, SLICES = THREADS / CH;  // chunks of a head; keys taken side by side
  __shared__ int last_kept[THREADS / 64];
  __shared__ uint64_t unseen;
  __shared__ float sums[SLICES][D];
  const int b = blockIdx.y, g = blockIdx.z, i0 = blockIdx.x * 64, tid = threadIdx.x, lane = tid & 63;
  const uint8_t *mask = key_mask + (long)b * len;
  auto lo = [&](int i) { return window <= 0 ? 0 : max(0, causal ? i - window + 1 : i - window); };
  auto hi = [&](int i) { return causal ? min(i + 1, num_k) : window > 0 ? min(i + window + 1, num_k) : num_k; };
  const int h0 = hi(i0);
  int last = -1;
  for (int k = h0 - 1 - tid; k >= lo(i0) && last < 0; k -= THREADS)
    if (mask[k]) last = k;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) last = max(last, __shfl_xor(last, off, 64));
  if (lane == 0) last_kept[tid >> 6] = last;
  __syncthreads();
  if (tid < 64) {
    for (int w = 0; w < THREADS / 64; ++w) last = max(last, last_kept[w]);
    const uint64_t next = __builtin_amdgcn_ballot_w64(h0 + lane < num_k && mask[min(h0 + lane, num_k - 1)] != 0);
    const int i = i0 + lane, n = hi(i) - h0;  // 0 <= n < 64
    const uint64_t below = next & ((1ull << n) - 1);
    if (below) last = h0 + 63 - __builtin_clzll(below);
    const uint64_t u = __builtin_amdgcn_ballot_w64(i < num_q && last < lo(i));
    if (lane == 0) unseen = u;
  }
  __syncthreads();
  const uint64_t rows = unseen;
  if (!rows) return;
  const int c = tid % CH, slice = tid / CH;
  const long vs = v_stride / VEC, os = o_stride / VEC;
  const CHUNK *v = V + (long)b * len * vs + g * CH + c;
  float part[VEC] = {};
  for (int k = slice; k < num_k; k += 8 * SLICES) {
    CHUNK t[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = v[min(k + e * SLICES, num_k - 1) * vs];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float f[VEC];
      widen(t[e], f);
      if (k + e * SLICES < num_k)
#pragma unroll
        for (int i = 0; i < VEC; ++i) part[i] += f[i];
    }
  }
#pragma unroll
  for (int i = 0; i < VEC; ++i) sums[slice][c * VEC + i] = part[i];
  __syncthreads();
  // every slice's threads then hold the chunk's mean, and write it to a share of the rows and query heads
  float mean[VEC] = {};
  for (int s = 0; s < SLICES; ++s)
#pragma unroll
    for (int i = 0; i < VEC; ++i) mean[i] += sums[s][c * VEC + i];
#pragma unroll
  for (int i = 0; i < VEC; ++i) mean[i] /= num_k;
  const CHUNK m = narrow(mean);
  const int group = hq / hkv;
  CHUNK *out = O + ((long)b * len + i0) * os + (long)g * group * CH + c;
  for (int t = slice; t < 64 * group; t += SLICES)
    if (rows >> (t / group) & 1) out[(t / group) * os + t % group * CH] = m;
}

// Thread t packs word t % words of sequence t / words: bit j <- key_mask[seq_start + 32 w + j] != 0 for keys
// inside the sequence, 0 past its length.
__global__ void __launch_bounds__(THREADS)
pack_key_bits_kernel(const uint8_t *__restrict__ key_mask, const int32_t *__restrict__ seq_start,
                     const int32_t *__restrict__ seq_len, int num_seqs, int max_seq_len, int words,
                     uint32_t *__restrict__ bits) {
  const long t = (long)blockIdx.x * THREADS + threadIdx.x;
  if (t >= (long)num_seqs * words) return;
  const int b = (int)(t / words), w = (int)(t % words);
  const int len = min(max(seq_len[b], 0), max_seq_len);
  const long start = seq_start[b];
  uint32_t word = 0;
  for (int j = 0; j < 32; ++j) {
    const int key = 32 * w + j;
    if (key < len && key_mask[start + key]) word |= 1u << j;
  }
  bits[t] = word;
}

}  // namespace

hipError_t dx_pack_key_bits_launch(const uint8_t *key_mask, const int32_t *seq_start, const int32_t *seq_len,
                                   int num_seqs, int max_seq_len, int words, uint32_t *bits, hipStream_t s) {
  const long total = (long)num_seqs * words;
  pack_key_bits_kernel<<<dim3((unsigned)((total + THREADS - 1) / THREADS)), dim3(THREADS), 0, s>>>(
      key_mask, seq_start, seq_len, num_seqs, max_seq_len, words, bits);
  return hipGetLastError();
}

hipError_t dx_attn_bf16(const AttnArgs &a, hipStream_t s) {
  switch (a.d) {
    case 64: return launch_bf16_d<64>(a, s);
    case 128: return launch_bf16_d<128>(a, s);
    case 256: return launch_bf16_d<256>(a, s);
  }
  return hipErrorInvalidValue;
}

hipError_t dx_attn_f32(const AttnArgs &a, hipStream_t s) {
  switch (a.d) {
    case 64: return launch_f32_d<64>(a, s);
    case 128: return launch_f32_d<128>(a, s);
    case 256: return launch_f32_d<256>(a, s);
  }
  return hipErrorInvalidValue;
}

hipError_t dx_vt_zero_tails_launch(uint16_t *vt, const int32_t *seq_len, const int32_t *vt_start, int num_seqs,
                                   int vt_rows, long vt_ld, hipStream_t s) {
  const dim3 grid((unsigned)num_seqs, (unsigned)((vt_rows + THREADS / 64 - 1) / (THREADS / 64)));
  vt_zero_tails_kernel<<<grid, dim3(THREADS), 0, s>>>(vt, seq_len, vt_start, vt_rows, vt_ld);
  return hipGetLastError();
}

hipError_t dx_transpose_v_launch(const uint16_t *v, uint16_t *vt, const int32_t *seq_start, const int32_t *seq_len,
                                 const int32_t *vt_start, long vt_seq_stride, int num_seqs, int max_seq_len, int hkv,
                                 int d, long v_stride, long vt_ld, hipStream_t s) {
  const dim3 grid((max_seq_len + 63) / 64, num_seqs, hkv * (d / 64));
  transpose_v_kernel<false><<<grid, dim3(THREADS), 0, s>>>(v, vt, seq_start, seq_len, vt_start, vt_seq_stride,
                                                          max_seq_len, d, v_stride, vt_ld, PaddedPrep{});
  return hipGetLastError();
}

hipError_t dx_prepare_padded_launch(const uint16_t *v, uint16_t *vt, const uint8_t *key_mask, uint32_t *bits,
                                    int32_t *seq_start, int32_t *seq_len, int batch, int len, int words, int hkv, int d,
                                    long v_stride, long vt_seq_stride, long vt_ld, hipStream_t s) {
  const dim3 grid((len + 63) / 64, batch, hkv * (d / 64) + 1);
  transpose_v_kernel<true><<<grid, dim3(THREADS), 0, s>>>(v, vt, nullptr, nullptr, nullptr, vt_seq_stride, len, d,
                                                         v_stride, vt_ld,
                                                         PaddedPrep{key_mask, bits, seq_start, seq_len, words});
  return hipGetLastError();
}

hipError_t dx_fill_unseen_launch(const AttnArgs &a, const uint8_t *key_mask, int num_q, int num_k, bool f32,
                                 hipStream_t s) {
  const dim3 grid((num_q + 63) / 64, a.num_seqs, a.hkv);
  auto run = [&](auto kern, auto chunk) {
    typedef decltype(chunk) CHUNK;
    kern<<<grid, dim3(THREADS), 0, s>>>(static_cast<const CHUNK *>(a.v), static_cast<CHUNK *>(a.out), key_mask,
                                        a.max_seq_len, num_q, num_k, a.hq, a.hkv, a.v_stride, a.out_stride, a.window,
                                        a.causal);
    return hipGetLastError();
  };
  switch (a.d) {
    case 64: return f32 ? run(fill_unseen_kernel<floatx4, 4, 64>, floatx4{}) : run(fill_unseen_kernel<u32x4, 8, 64>, u32x4{});
    case 128:
      return f32 ? run(fill_unseen_kernel<floatx4, 4, 128>, floatx4{}) : run(fill_unseen_kernel<u32x4, 8, 128>, u32x4{});
    case 256:
      return f32 ? run(fill_unseen_kernel<floatx4, 4, 256>, floatx4{}) : run(fill_unseen_kernel<u32x4, 8, 256>, u32x4{});
  }
  return hipErrorInvalidValue;
}
