// Clef joint schema head on gfx950, fp32 (the reference's head runs in the model dtype; its
// fixture and this path are fp32). The steps of src/deciax/models/clef/head.py:54-111 map onto a
// few kernels that the host driver (deciax_amd/clef_head.py) chains:
//   layer_norm_f32   nn.py:22-29 / head.py:20-21            one wave per row
//   linear_f32       nn.py:11-19 + text.py:21-22, + exact GELU and residual accumulate
//   span_means_f32   head.py:24-29                          one workgroup per span
//   mha_f32          head.py:41-51 core: masked softmax(q k^T / sqrt(dh)) v, blocked.py:9-32
//   gather_rows_f32  head.py:32-33                          (optionally accumulating)
//   routing_f32      head.py:76-85: per-question softmax over owned options and the summary
//   fields_init_f32  head.py:86-88
//   features_f32     head.py:97-106: anchor / prior, cosine, [f, o, f*o, |f-o|]
//   combine_f32      head.py:107-111
// Long memories make the projections of their rows the head's cost (8 x 4096 tokens: 7 of 8.9 ms), a single request
// the latency of some sixty small launches.
#include "common.h"
#include "kernels.h"
#include "loads.h"

namespace {

constexpr int THREADS = 256;
constexpr float MASK_FILL = -1e30f;  // src/deciax/kernels/attention/reference.py:8

DX_DEVICE float wave_reduce_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
DX_DEVICE float wave_reduce_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// Sum / max over the 256 threads of a workgroup (every thread gets the result).
DX_DEVICE float block_sum(float v, float *red) {
  v = wave_reduce_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}
// Several sums at once: two barriers for all of them.
template <int N>
DX_DEVICE void block_sums(float (&v)[N], float (*red)[THREADS / 64]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = wave_reduce_sum(v[i]);
  __syncthreads();
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < N; ++i) red[i][w] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = red[i][0] + red[i][1] + red[i][2] + red[i][3];
}
DX_DEVICE float block_max(float v, float *red) {
  v = wave_reduce_max(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

DX_DEVICE float gelu_erf(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

// y = (x - mean) / sqrt(mean((x - mean)^2) + eps) * w + b, one wave per row.
__global__ void __launch_bounds__(THREADS)
layer_norm_f32_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ b,
                      float *__restrict__ y, long rows, int d, long ldx, long ldy, float eps) {
  const long row = (long)blockIdx.x * (THREADS / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const float *xr = x + row * ldx;
  float s = 0.f;
  for (int i = lane; i < d; i += 64) s += xr[i];
  const float mean = wave_reduce_sum(s) / (float)d;
  float q = 0.f;
  for (int i = lane; i < d; i += 64) {
    const float z = xr[i] - mean;
    q += z * z;
  }
  const float r = 1.0f / sqrtf(wave_reduce_sum(q) / (float)d + eps);
  float *yr = y + row * ldy;
  for (int i = lane; i < d; i += 64) yr[i] = (xr[i] - mean) * r * w[i] + (b ? b[i] : 0.f);
}

// The same with the row in registers (16-byte chunk c = lane + 64 i), so it is read once and all of it at once:
// d <= 256 MAXC, a multiple of 4, rows and weights 16-byte aligned.
template <int MAXC>
__global__ void __launch_bounds__(THREADS)
layer_norm_f32_row_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ b,
                          float *__restrict__ y, long rows, int d, long ldx, long ldy, float eps) {
  const long row = (long)blockIdx.x * (THREADS / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63, nch = d / 4;
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  const floatx4 *xr = reinterpret_cast<const floatx4 *>(x + row * ldx);
  floatx4 v[MAXC];
#pragma unroll
  for (int i = 0; i < MAXC; ++i) v[i] = lane + 64 * i < nch ? xr[lane + 64 * i] : zero;
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < MAXC; ++i) s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
  const float mean = wave_reduce_sum(s) / (float)d;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < MAXC; ++i)
    if (lane + 64 * i < nch) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[i][e] -= mean;
        q += v[i][e] * v[i][e];
      }
    }
  const float r = 1.0f / sqrtf(wave_reduce_sum(q) / (float)d + eps);
  floatx4 *yr = reinterpret_cast<floatx4 *>(y + row * ldy);
#pragma unroll
  for (int i = 0; i < MAXC; ++i) {
    const int c = lane + 64 * i;
    if (c < nch) {
      const floatx4 wc = reinterpret_cast<const floatx4 *>(w)[c];
      const floatx4 bc = b ? reinterpret_cast<const floatx4 *>(b)[c] : zero;
      yr[c] = v[i] * r * wc + bc;
    }
  }
}

// fp32 products on the matrix core: v_mfma_f32_16x16x4_f32 (fp32 products and sums, 256 FLOP per cycle and
// CU). Lane l supplies A row (l % 16) and B column (l % 16) at contraction index l / 16, and gets back column
// l % 16, rows (l / 16) * 4 + r. Which four contraction indices meet in one MFMA is free, so a lane takes runs of
// consecutive ones: its operands are 16-byte loads straight from global memory, no LDS.
DX_DEVICE floatx4 mfma16_f32(float a, float b, floatx4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// y[m, n] = (acc ? y[m, n] : 0) + act(x[m, :] . w[n, :] + bias[n]); act: 0 identity, 1 exact GELU.
// Rows that are not whole 16-byte chunks, and short ones (the others take the split products below). A workgroup
// computes 16 TM x 16 TN outputs; its KW waves split k in runs of 32 (interleaved, so together they read whole cache
// lines) and add their sums through LDS, in the same order for every tile shape, so that a row does not depend on m.
// A wave's lane (l % 16, l / 16) holds k values k0 + 16 c + 4 (l / 16) .. + 3 of its row, for chunks c < KC, loaded one
// step ahead into the other half of its registers. Rows past m and n read the last row (not stored). VEC: rows are
// 16-byte aligned, else elements are read one at a time.
template <int TM, int TN, bool VEC>
__global__ void __launch_bounds__(256)
linear_f32_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
                  float *__restrict__ y, long m, int n, int k, long ldx, long ldw, long ldy, int act, int acc) {
  constexpr int KW = 4, KC = 2, STEP = 16 * KC;
  const int tid = threadIdx.x, lane = tid & 63, kw = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const unsigned num_n = (n + 16 * TN - 1) / (16 * TN);
  const long m0 = (long)(blockIdx.x / num_n) * (16 * TM);
  const int n0 = (int)(blockIdx.x % num_n) * (16 * TN);
  const float *xp[TM], *wp[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) xp[i] = x + min(m0 + 16 * i + lr, m - 1) * ldx + 4 * lk;
#pragma unroll
  for (int j = 0; j < TN; ++j) wp[j] = w + (long)min(n0 + 16 * j + lr, n - 1) * ldw + 4 * lk;

  auto load4 = [&](const float *p) __attribute__((always_inline)) {
    if constexpr (VEC) {
      return *reinterpret_cast<const floatx4 *>(p);
    } else {
      const floatx4 v = {p[0], p[1], p[2], p[3]};
      return v;
    }
  };
  floatx4 c[TM][TN] = {};
  floatx4 a0[TM][KC], b0[TN][KC], a1[TM][KC], b1[TN][KC];
  // a whole step at kk
  auto load = [&](floatx4 (&a)[TM][KC], floatx4 (&b)[TN][KC], int kk) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < KC; ++s) {
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i][s] = load4(xp[i] + kk + 16 * s);
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j][s] = load4(wp[j] + kk + 16 * s);
    }
  };
  auto part4 = [&](const float *p, int left) __attribute__((always_inline)) {  // the first `left` of 4, then zeros
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < left) v[e] = p[e];
    return v;
  };
  auto mma = [&](const floatx4 (&a)[TM][KC], const floatx4 (&b)[TN][KC]) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < KC; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) c[i][j] = mfma16_f32(a[i][s][e], b[j][s][e], c[i][j]);
  };
  // whole steps kw, kw + KW, ... (the prefetch past the last reloads it), then the partial one, if any
  const int full = k / STEP;
  const int mine = full > kw ? (full - kw - 1) / KW + 1 : 0;
  auto at = [&](int t) { return (kw + min(t, mine - 1) * KW) * STEP; };
  if (mine > 0) {
    load(a0, b0, at(0));
    int t = 0;
    for (; t + 1 < mine; t += 2) {
      load(a1, b1, at(t + 1));
      __builtin_amdgcn_sched_barrier(0);  // the next step's loads go out before this step's products
      mma(a0, b0);
      load(a0, b0, at(t + 2));
      __builtin_amdgcn_sched_barrier(0);
      mma(a1, b1);
    }
    if (t < mine) mma(a0, b0);
  }
  if (k % STEP && kw == full % KW) {
    const int kk = full * STEP;
#pragma unroll
    for (int s = 0; s < KC; ++s) {
      const int left = k - kk - 16 * s - 4 * lk;
#pragma unroll
      for (int i = 0; i < TM; ++i) a0[i][s] = part4(xp[i] + kk + 16 * s, left);
#pragma unroll
      for (int j = 0; j < TN; ++j) b0[j][s] = part4(wp[j] + kk + 16 * s, left);
    }
    mma(a0, b0);
  }

  auto store = [&](long gm, int gn, float v) __attribute__((always_inline)) {
    if (gm >= m || gn >= n) return;
    v += bias ? bias[gn] : 0.f;
    if (act == 1) v = gelu_erf(v);
    float *dst = y + gm * ldy + gn;
    *dst = acc ? *dst + v : v;
  };
  constexpr int TILE = 256 * TM * TN;
  __shared__ float part[KW * TILE];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[kw * TILE + (16 * i + 4 * lk + r) * (16 * TN) + 16 * j + lr] = c[i][j][r];
  __syncthreads();
  for (int idx = tid; idx < TILE; idx += 256) {
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < KW; ++q) v += part[q * TILE + idx];
    store(m0 + idx / (16 * TN), n0 + idx % (16 * TN), v);
  }
}

// fp32 operands as sums of three bf16 (x = h + m + l, each the bf16 nearest to what is left: 24 bits or more),
// multiplied by six bf16 MFMAs: h h into one fp32 accumulator, l h, h l, m m, m h, h m into another, 2^-8 of its size,
// so that one rounding per 16 k counts. What is left out (m l, l m, l l) is below 2^-24 of |x w| (m below 2^-8 |x|, l
// below 2^-17 |x|, so 2^-25 for each of the first two): the rounding of an fp32 product at most. The pair of accumulators
// joins the sum after every PART k. Error against 64 bits at k = 1024 / 4096: 1.0e-7 / 1.2e-7 (over all of k 1.9e-7 /
// 4.0e-7; both accumulators in one 3.4e-7 / 7.2e-7; fp32 MFMAs in one chain 4.0e-7 / 8.2e-7, in four 2.9e-7 / 5.7e-7).
// Two kernels, the same chain of MFMAs and sums for an output in both, so that a row does not depend on m.
// Some outputs, and no others, are multiplied again with fp32 MFMAs: those that are not finite (an infinity, a NaN or a
// value past the largest bf16 leaves its row or column so, inf - inf), and those below 2^-84. bf16 has fp32's exponents, so
// an operand below 2^-109 loses bits of l (error 2.7e-6 at 1e-35, 2.7e-4 at 1e-37), and its row's outputs are that small
// unless the other operand is past 2^24 / k.
constexpr int PART = 256;

DX_DEVICE bool outside_split(float v) { return !(fabsf(v) < INFINITY) || (fabsf(v) < 0x1p-84f && v != 0.f); }

DX_DEVICE void split3(const floatx4 &v, u32x2 (&p)[3]) {
  float a[4] = {v[0], v[1], v[2], v[3]};
#pragma unroll
  for (int t = 0; t < 3; ++t) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t w = pack_bf2(a[2 * i], a[2 * i + 1]);
      p[t][i] = w;
      if (t < 2) {
        a[2 * i] -= lo_bf(w);
        a[2 * i + 1] -= hi_bf(w);
      }
    }
  }
}

// One lane's outputs of a 32 x 32 block, from the rows of x and w that the lane feeds (whole 16-byte chunks). Rare, so
// a plain loop.
DX_DEVICE floatx16 product32_f32(const float *xr, const float *wr, int k, int lhalf) {
  floatx16 c;
#pragma unroll
  for (int r = 0; r < 16; ++r) c[r] = 0.f;
  for (int k0 = 4 * lhalf; k0 < k + 4 * lhalf; k0 += 8) {  // both lane halves take as many steps
    floatx4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
    if (k0 < k) {
      a = *reinterpret_cast<const floatx4 *>(xr + k0);
      b = *reinterpret_cast<const floatx4 *>(wr + k0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(b[e], a[e], c, 0, 0, 0);
  }
  return c;
}

// Four sums of a row, columns col..col + 3 at dst: bias, act and accumulation as linear_f32_kernel.
DX_DEVICE void store_quad(floatx4 v, float *dst, const float *__restrict__ bias, int col, int n, int act, int acc_y,
                          int vec_y) {
  if (vec_y && col + 4 <= n) {
    if (bias) v += *reinterpret_cast<const floatx4 *>(bias + col);
    if (act == 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gelu_erf(v[e]);
    }
    if (acc_y) v += *reinterpret_cast<const floatx4 *>(dst);
    *reinterpret_cast<floatx4 *>(dst) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (col + e >= n) continue;
      float s = v[e] + (bias ? bias[col + e] : 0.f);
      if (act == 1) s = gelu_erf(s);
      dst[e] = acc_y ? dst[e] + s : s;
    }
  }
}

// 16 bytes per lane from a buffer resource into LDS at lds + 16 * lane. The builtin is compiled in the device pass only:
// this clang drops a kernel's host-side symbols when the host pass sees it.
typedef __attribute__((address_space(3))) void lds_void;
DX_DEVICE void lds_load16(__amdgpu_buffer_rsrc_t rsrc, float *lds, int voffset) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void *)lds, 16, voffset, 0, 0, 0);
#endif
}

// Few rows, or few columns: tiles of 32 x 32, a part of k per wave (parts w, w + WAVES, .. for wave w). A wave streams
// SK columns of its 64 rows at a time through a ring of its own in LDS (loads to LDS, no barrier: a load straight into
// the MFMA layout would take four rows per quad of lanes and four times the address cycles; 11 us for 8 at 23 x 1024 x
// 1024, 35 for 22 at k = 4096), reads them in the MFMA layout (lane (l % 32, l / 32): k 8 (l / 32) .. + 7 of row l % 32)
// and splits them itself. The parts' sums meet in LDS. What bounds it: some 110 vector instructions a wave and 16 k.
template <int WAVES, int SK, int RING>
__global__ void __launch_bounds__(64 * WAVES)
linear_split_small_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
                          float *__restrict__ y, long m, int n, int k, long ldx, long ldw, long ldy, int act, int acc_y,
                          int vec_y) {
  constexpr int STAGES = PART / SK, SUB = SK / 16;      // stages of a part; 16 k of a stage
  constexpr int CPR = SK / 4, RPI = 64 / CPR, NI = 32 / RPI;  // 16-byte chunks per row; rows and instructions per load
  constexpr int SLOT = 64 * SK;                         // floats: x's 32 rows, then w's
  static_assert((SK == 16 || SK == 32) && STAGES % 2 == 0 && WAVES >= 4 && (RING - 1) * 2 * NI <= 63, "wave schedule");
  // the rings, then the waves' sums; a flag over the first ring at the end. One array: with several the compiler waits for
  // every load to LDS before each read of the ring.
  __shared__ __attribute__((aligned(1024))) float smem[WAVES * RING * SLOT + WAVES * 1024];
  floatx4(*const sums)[4][64] = reinterpret_cast<floatx4(*)[4][64]>(smem + WAVES * RING * SLOT);  // [register / 4][lane]
  int *const bad = reinterpret_cast<int *>(smem);
  const int num_n = (n + 31) / 32;
  const long m0 = (long)(blockIdx.x / num_n) * 32;
  const int n0 = (int)(blockIdx.x % num_n) * 32;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int arows = (int)min(32L, m - m0), brows = min(32, n - n0);
  // rows past m and n, and columns past k, read as zeros
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(x + m0 * ldx), (short)0, (int)(((long)(arows - 1) * ldx + k) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(w + (long)n0 * ldw), (short)0, (int)(((long)(brows - 1) * ldw + k) * 4), 0x00020000);
  const int parts = (k + PART - 1) / PART, rounds = (parts + WAVES - 1) / WAVES;
  // Row r's chunk c lies in slot c ^ swz(r): 16 rows' reads of one chunk fall on all banks
  auto swz = [](int r) { return SK == 32 ? (r >> 1) & 7 : (r >> 2) & 3; };
  float *const mine = smem + wave * RING * SLOT;
  int col[NI], xoff[NI], woff[NI];  // of the lane's 16 bytes in each instruction
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int row = j * RPI + lane / CPR;
    col[j] = 4 * ((lane % CPR) ^ swz(row));
    xoff[j] = (int)(row * ldx * 4);
    woff[j] = (int)(row * ldw * 4);
  }
  auto load = [&](int u) __attribute__((always_inline)) {  // the wave's stage u
    const int c0 = ((u / STAGES) * WAVES + wave) * PART + u % STAGES * SK;
    float *to = mine + u % RING * SLOT;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int at = column_offset(c0 + col[j], k, (c0 + col[j]) * 4);
      lds_load16(rx, to + j * 256, xoff[j] + at);
      lds_load16(rw, to + 32 * SK + j * 256, woff[j] + at);
    }
  };
  auto read = [&](floatx4 (&v)[SUB][4], int u) __attribute__((always_inline)) {
    const float *from = mine + u % RING * SLOT + lrow * SK;
#pragma unroll
    for (int i = 0; i < SUB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int at = ((4 * i + 2 * lhalf + j) ^ swz(lrow)) * 4;
        v[i][j] = *reinterpret_cast<const floatx4 *>(from + at);
        v[i][2 + j] = *reinterpret_cast<const floatx4 *>(from + 32 * SK + at);
      }
  };
  auto planes = [&](const floatx4 &lo, const floatx4 &hi, bf16x8 (&f)[3]) __attribute__((always_inline)) {
    u32x2 p[3], q[3];
    split3(lo, p);
    split3(hi, q);
#pragma unroll
    for (int t = 0; t < 3; ++t) f[t] = as_bf16x8(u32x4{p[t][0], p[t][1], q[t][0], q[t][1]});
  };
  floatx16 c, small;
  struct Planes {
    bf16x8 a[3], b[3];
  };
  // multiplies 16 k while the next 16 are split, the vector instructions spread over the MFMAs
  auto step = [&](const Planes &p, const floatx4 (&next)[4], Planes &q) __attribute__((always_inline)) {
    small = mfma32(p.b[0], p.a[2], small);
    c = mfma32(p.b[0], p.a[0], c);
    small = mfma32(p.b[2], p.a[0], small);
    small = mfma32(p.b[1], p.a[1], small);
    small = mfma32(p.b[0], p.a[1], small);
    small = mfma32(p.b[1], p.a[0], small);
    planes(next[0], next[1], q.a);
    planes(next[2], next[3], q.b);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // stage u has landed once the RING - 1 younger ones are all that is in flight
  auto landed = [&]() __attribute__((always_inline)) {
    constexpr int VM = (RING - 1) * 2 * NI;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4) << 14 | 7 << 4 | 15 << 8);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto refill = [&](int u) __attribute__((always_inline)) {  // stage u's slot, read by now, takes stage u + RING
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(15 | 3 << 14 | 7 << 4);
    __builtin_amdgcn_sched_barrier(0);
    load(u + RING);
    __builtin_amdgcn_sched_barrier(0);
  };
  floatx4 total = {0.f, 0.f, 0.f, 0.f};  // of the first four waves: registers 4 wave .. + 3 of lane
  // Stage u + 1 (SK 32) or u + 2 (SK 16) is read while stage u is multiplied.
  floatx4 v0[SUB][4], v1[SUB][4];
  Planes p0, p1;
  if (wave < parts) {
#pragma unroll
    for (int i = 0; i < RING; ++i) load(i);
    landed();
    read(v0, 0);
    refill(0);
    planes(v0[0][0], v0[0][1], p0.a);
    planes(v0[0][2], v0[0][3], p0.b);
    if constexpr (SUB == 1) {
      landed();
      read(v1, 1);
      refill(1);
    }
  }
  for (int r = 0; r < rounds; ++r) {
#pragma unroll
    for (int e = 0; e < 16; ++e) c[e] = small[e] = 0.f;
    if (r * WAVES + wave < parts) {
      for (int t = 0; t < STAGES; t += 2) {
        const int u = r * STAGES + t;
        if constexpr (SUB == 1) {
          landed();
          read(v0, u + 2);
          __builtin_amdgcn_sched_barrier(0);
          step(p0, v1[0], p1);
          refill(u + 2);
          landed();
          read(v1, u + 3);
          __builtin_amdgcn_sched_barrier(0);
          step(p1, v0[0], p0);
          refill(u + 3);
        } else {
          landed();
          read(v1, u + 1);
          __builtin_amdgcn_sched_barrier(0);
          step(p0, v0[SUB - 1], p1);
          refill(u + 1);
          step(p1, v1[0], p0);
          landed();
          read(v0, u + 2);
          __builtin_amdgcn_sched_barrier(0);
          step(p0, v1[SUB - 1], p1);
          refill(u + 2);
          step(p1, v0[0], p0);
        }
      }
    }
    if (r > 0) __syncthreads();  // the last round's sums are read
#pragma unroll
    for (int q = 0; q < 4; ++q)
      sums[wave][q][lane] = floatx4{c[4 * q] + small[4 * q], c[4 * q + 1] + small[4 * q + 1], c[4 * q + 2] + small[4 * q + 2],
                                    c[4 * q + 3] + small[4 * q + 3]};
    __syncthreads();
    if (wave < 4)
      for (int q = 0; q < min(WAVES, parts - r * WAVES); ++q) total += sums[q][wave][lane];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // loads to LDS past the last part
  if (tid == 0) *bad = 0;
  __syncthreads();
  if (wave < 4)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (outside_split(total[e])) *bad = 1;
  __syncthreads();
  const long row = m0 + lrow;
  if (*bad) {
    if (wave == 0) {
      const floatx16 f = product32_f32(x + min(row, m - 1) * ldx, w + (long)min(n0 + lrow, n - 1) * ldw, k, lhalf);
#pragma unroll
      for (int q = 0; q < 4; ++q) sums[0][q][lane] = floatx4{f[4 * q], f[4 * q + 1], f[4 * q + 2], f[4 * q + 3]};
    }
    __syncthreads();
    if (wave < 4) {
      const floatx4 f = sums[0][wave][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) total[e] = outside_split(total[e]) ? f[e] : total[e];
    }
  }
  if (wave < 4 && row < m) {
    const int col = n0 + 8 * wave + 4 * lhalf;
    store_quad(total, y + row * ldy + col, bias, col, n, act, acc_y, vec_y);
  }
}

// Many rows: tile (64 TM) x (64 TN) of 2 x 2 waves, 16 k per step. A step's fp32 chunks arrive in registers one step
// ahead, are split once per workgroup and go to the other half of the LDS. What bounds it: the bf16 MFMAs, 6 / 16 of
// the cycles of fp32 ones, at the rate the large bf16 GEMMs reach (1.2 PFLOP/s of them). Two register sets, or the
// split spread between the MFMAs, measured the same or slower; 32 k per step 20% slower.
template <int TM, int TN>
__global__ void __launch_bounds__(256, 2)
linear_split_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
                    float *__restrict__ y, long m, int n, int k, long ldx, long ldw, long ldy, int act, int acc_y,
                    int vec_y) {
  constexpr int BM = 64 * TM, BN = 64 * TN, ROWS = BM + BN, BK = 16;
  constexpr int CPR = BK / 4, RPP = 256 / CPR;          // 16-byte chunks per row; rows per pass of the workgroup
  constexpr int AP = BM / RPP, BP = BN / RPP;           // chunks per thread
  // planes [h, m, l][k / 8][row][8]: fragment reads run over consecutive rows, and the two halves of a write's rows
  // fall on different banks (+3% over [row][16])
  constexpr int HALF = ROWS * 8 + 64, PLANE = 2 * HALF, STAGE = 3 * PLANE;  // bf16 elements
  __shared__ __attribute__((aligned(1024))) uint16_t smem[2 * STAGE];

  const int num_n = (n + BN - 1) / BN, nblocks = gridDim.x;
  // each XCD (workgroups go round-robin over 8) takes a contiguous run of tiles, the tiles of one row block together
  const int per = nblocks / 8, rem = nblocks % 8, xcd = blockIdx.x % 8, idx = blockIdx.x / 8;
  const int tile = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
  const long m0 = (long)(tile / num_n) * BM;
  const int n0 = tile % num_n * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, lrow = lane & 31, lhalf = lane >> 5;
  const int arows = (int)min((long)BM, m - m0), brows = min(BN, n - n0);
  // rows past m and n read as zeros
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(x + m0 * ldx), (short)0, (int)(((long)(arows - 1) * ldx + k) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(w + (long)n0 * ldw), (short)0, (int)(((long)(brows - 1) * ldw + k) * 4), 0x00020000);
  const int prow = tid / CPR, pc = tid % CPR;
  const int xoff = (int)((prow * ldx + 4 * pc) * 4), woff = (int)((prow * ldw + 4 * pc) * 4);
  const int xstep = (int)(RPP * ldx * 4), wstep = (int)(RPP * ldw * 4);
  floatx4 st[AP + BP];
  auto load = [&](int kk) __attribute__((always_inline)) {
    const int at = column_offset(kk + 4 * pc, k, kk * 4);  // chunks at k or past it read as zeros
#pragma unroll
    for (int j = 0; j < AP; ++j)
      st[j] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rx, xoff + j * xstep + at, 0, 0));
#pragma unroll
    for (int j = 0; j < BP; ++j)
      st[AP + j] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rw, woff + j * wstep + at, 0, 0));
  };
  const int dst = pc / 2 * HALF + prow * 8 + pc % 2 * 4;
  auto put = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < AP + BP; ++j) {
      u32x2 p[3];
      split3(st[j], p);
      uint16_t *d = smem + stage * STAGE + dst + (j < AP ? j * RPP : BM + (j - AP) * RPP) * 8;
#pragma unroll
      for (int t = 0; t < 3; ++t) *reinterpret_cast<u32x2 *>(d + t * PLANE) = p[t];
    }
  };
  floatx16 c[TM][TN], small[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) c[i][j][r] = small[i][j][r] = total[i][j][r] = 0.f;
  auto fold = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          total[i][j][r] += c[i][j][r] + small[i][j][r];
          c[i][j][r] = small[i][j][r] = 0.f;
        }
  };
  auto mma = [&](int stage) __attribute__((always_inline)) {
    const uint16_t *pa = smem + stage * STAGE + lhalf * HALF + (wm * 32 * TM + lrow) * 8;
    const uint16_t *pb = smem + stage * STAGE + lhalf * HALF + (BM + wn * 32 * TN + lrow) * 8;
    bf16x8 a[3][TM], b[3][TN];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
#pragma unroll
      for (int i = 0; i < TM; ++i) a[t][i] = as_bf16x8(*reinterpret_cast<const u32x4 *>(pa + t * PLANE + 32 * i * 8));
#pragma unroll
      for (int j = 0; j < TN; ++j) b[t][j] = as_bf16x8(*reinterpret_cast<const u32x4 *>(pb + t * PLANE + 32 * j * 8));
    }
    constexpr int PA[6] = {0, 2, 0, 1, 1, 0}, PB[6] = {0, 0, 2, 1, 0, 1};
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          floatx16 &acc = t == 0 ? c[i][j] : small[i][j];
          acc = mfma32(b[PB[t]][j], a[PA[t]][i], acc);
        }
  };
  const int steps = (k + BK - 1) / BK;
  load(0);
  put(0);
  load(min(BK, (steps - 1) * BK));
  __syncthreads();
  for (int t = 0; t < steps; ++t) {
    mma(t & 1);
    // (where the fold stands decides the registers: here 128 x 128 tiles keep two workgroups a CU, and after the barrier
    // 128 x 64 tiles let the split run beside the MFMAs, 33 us for 39 at k = 1024)
    if constexpr (TN == 2)
      if ((t + 1) % (PART / BK) == 0 || t + 1 == steps) fold();
    put((t + 1) & 1);  // past the end: old chunks that nothing reads
    load(min(t + 2, steps - 1) * BK);
    __syncthreads();
    if constexpr (TN == 1)
      if ((t + 1) % (PART / BK) == 0 || t + 1 == steps) fold();
  }

  bool bad = false;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        bad = bad || outside_split(total[i][j][r]);
      }
  if (__builtin_amdgcn_ballot_w64(bad)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const floatx16 f = product32_f32(x + min(m0 + wm * 32 * TM + 32 * i + lrow, m - 1) * ldx,
                                         w + (long)min(n0 + wn * 32 * TN + 32 * j + lrow, n - 1) * ldw, k, lhalf);
#pragma unroll
        for (int r = 0; r < 16; ++r) total[i][j][r] = outside_split(total[i][j][r]) ? f[r] : total[i][j][r];
      }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const long row = m0 + wm * 32 * TM + 32 * i + lrow;
    if (row >= m) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = n0 + wn * 32 * TN + 32 * j + 8 * q + 4 * lhalf;
        const floatx16 &v = total[i][j];
        store_quad(floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]}, y + row * ldy + col, bias, col, n, act, acc_y,
                   vec_y);
      }
    }
  }
}

// out[b * O + o, :] = mean of x[b * S + s, :] over s in [spans[b, o, 0], spans[b, o, 1]) (within
// [0, S)); an empty span gives 0 (head.py:28 divides by max(count, 1)). One workgroup per span and 256 columns.
// With `index`, row s of batch row b is x[index[b * S + s]] of a table of R rows: 48653 ids over 4096 spans, width
// 4096, take one pass over the rows they name (a gathered copy first: 346 us for it and 120 for its means).
template <bool GATHER>
__global__ void __launch_bounds__(THREADS)
span_means_f32_kernel(const float *__restrict__ x, const int32_t *__restrict__ index, const int32_t *__restrict__ spans,
                      float *__restrict__ out, int R, int S, int O, int d, long ldx, long ldo) {
  const int bo = blockIdx.x, b = bo / O, i = blockIdx.y * THREADS + threadIdx.x;
  const int lo = max(spans[2 * bo], 0), hi = min(spans[2 * bo + 1], S);
  if (i >= d) return;
  const float inv = 1.0f / (float)max(hi - lo, 1);
  auto row = [&](int s) __attribute__((always_inline)) {
    if constexpr (GATHER) return (long)min(max(index[(long)b * S + s], 0), R - 1);
    else return (long)b * S + s;
  };
  float s = 0.f;
  int t = lo;
  for (; t + 8 <= hi; t += 8) {  // eight rows in flight, added in order
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = x[row(t + e) * ldx + i];
#pragma unroll
    for (int e = 0; e < 8; ++e) s += v[e];
  }
  if (t < hi) {
    float v[7];
#pragma unroll
    for (int e = 0; e < 7; ++e) v[e] = x[row(min(t + e, hi - 1)) * ldx + i];
#pragma unroll
    for (int e = 0; e < 7; ++e)
      if (t + e < hi) s += v[e];
  }
  out[(long)bo * ldo + i] = hi > lo ? s * inv : 0.f;
}

// One workgroup per (b, query, head): scores over the K keys of batch row b into LDS, masked keys at
// MASK_FILL, softmax in fp32, then out = sum_k p_k v_k. q, k, v, out: rows of ld* floats, head h at
// columns [h dh, h dh + dh). key_mask: [B, K] bytes (nonzero = visible).
__global__ void __launch_bounds__(THREADS)
mha_f32_kernel(const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
               const uint8_t *__restrict__ key_mask, float *__restrict__ out, int Q, int K, int H, int dh, long ldq,
               long ldk, long ldv, long ldo) {
  extern __shared__ float smem[];  // K scores, then THREADS partial sums
  __shared__ float red[4];
  const int h = blockIdx.x % H, qi = (blockIdx.x / H) % Q, b = blockIdx.x / (H * Q);
  const float *qr = q + ((long)b * Q + qi) * ldq + (long)h * dh;
  const float scale = 1.0f / sqrtf((float)dh);
  float mx = MASK_FILL;
  for (int j = threadIdx.x; j < K; j += THREADS) {
    const float *kr = k + ((long)b * K + j) * ldk + (long)h * dh;
    float s = 0.f;
    for (int i = 0; i < dh; ++i) s = fmaf(qr[i], kr[i], s);
    s = key_mask[(long)b * K + j] ? s * scale : MASK_FILL;
    smem[j] = s;
    mx = fmaxf(mx, s);
  }
  mx = block_max(mx, red);
  float sum = 0.f;
  for (int j = threadIdx.x; j < K; j += THREADS) {
    const float p = expf(smem[j] - mx);
    smem[j] = p;
    sum += p;
  }
  sum = block_sum(sum, red);  // its barriers also publish the probabilities
  // dimensions [d0, d0 + dsub) per pass; thread t takes dimension d0 + t % dsub and keys t / dsub,
  // t / dsub + slices, ...; the slices' partial sums meet in LDS
  const int dsub = min(dh, THREADS), slices = THREADS / dsub;
  float *part = smem + K;
  for (int d0 = 0; d0 < dh; d0 += dsub) {
    const int i = d0 + (int)threadIdx.x % dsub, sl = (int)threadIdx.x / dsub;
    float acc = 0.f;
    if (i < dh && sl < slices)
      for (int j = sl; j < K; j += slices) acc = fmaf(smem[j], v[((long)b * K + j) * ldv + (long)h * dh + i], acc);
    part[threadIdx.x] = acc;
    __syncthreads();
    if ((int)threadIdx.x < min(dsub, dh - d0)) {
      float t = 0.f;
      for (int s2 = 0; s2 < slices; ++s2) t += part[s2 * dsub + threadIdx.x];
      out[((long)b * Q + qi) * ldo + (long)h * dh + d0 + threadIdx.x] = t / sum;
    }
    __syncthreads();
  }
}

// The same on the matrix core, head_dim D = 16 N <= 128, 16-byte aligned rows. A workgroup takes 16 QB queries of
// one (b, head); its WAVES waves take 16 SUB-key blocks in turn, each with its own running max m, row sum l and O,
// merged through LDS at the end (no barrier in the key loop). Layouts (see mfma16_f32):
//   S^T = K Q^T   contraction over head dims: lane (r, g) = (l % 16, l / 16) holds dims [4 N g, 4 N g + 4 N) of key
//                 row r and of query r, MFMA j contracting dim 4 N g + j of the four groups. It gets back query r,
//                 keys 4 g + 0..3 of the 16.
//   O^T += V^T P^T MFMA t contracts keys 4 g + t, whose probabilities the lane already holds; V rows come as N
//                 consecutive floats [N r, N r + N) of key 4 g + t, block c (c < N) taking float c, so the lane
//                 ends up with the 4 N consecutive dims [4 N g, 4 N g + 4 N) of query r.
// K of the next block is requested as soon as this block's scores are done, V at the start of its block.
template <int N>
DX_DEVICE void load_run(float (&v)[N], const float *p) {  // N consecutive floats, aligned as far as N allows
  if constexpr (N % 4 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 4) {
      const floatx4 t = *reinterpret_cast<const floatx4 *>(p + i);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i + e] = t[e];
    }
  } else if constexpr (N % 2 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 2) {
      const float2 t = *reinterpret_cast<const float2 *>(p + i);
      v[i] = t.x;
      v[i + 1] = t.y;
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = p[i];
  }
}

// e^d for d <= 0 (or NaN), within some two units in the last place: 2^n 2^f with n the integer nearest to d log2(e) and f
// what is left, log2(e) in two parts (Cody and Waite's reduction). expf without its tests for large results: 8 vector
// instructions for 13. Below the smallest number f, or the scaling by 2^n, ends in 0.
DX_DEVICE float exp_below0(float d) {
  constexpr double LOG2E = 1.4426950408889634074;
  constexpr float HI = (float)LOG2E, LO = (float)(LOG2E - (double)HI);
  const float n = rintf(fmaxf(d * HI, -300.f));
  const float f = __builtin_fmaf(d, LO, __builtin_fmaf(d, HI, -n));
  return ldexpf(fast_exp2(f), (int)n);
}

template <int N, int QB, int WAVES, int SUB>
__global__ void __launch_bounds__(64 * WAVES)
mha_f32_mfma_kernel(const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
                    const uint8_t *__restrict__ key_mask, float *__restrict__ out, int Q, int K, long ldq, long ldk,
                    long ldv, long ldo) {
  constexpr int D = 16 * N, KB = 16 * SUB;
  constexpr float NONE = -3e38f;  // running max before any key: below MASK_FILL
  __shared__ float os[WAVES][16 * QB][D + 4];
  __shared__ float ms[WAVES][16 * QB], ls[WAVES][16 * QB];
  const int h = blockIdx.y, b = blockIdx.z, q0 = blockIdx.x * 16 * QB;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const float scale = 1.0f / sqrtf((float)D);
  const float *kb = k + (long)b * K * ldk + (long)h * D + 4 * N * g;
  const float *vb = v + (long)b * K * ldv + (long)h * D + N * r16;
  const uint8_t *mb = key_mask + (long)b * K;

  float qf[QB][4 * N];
#pragma unroll
  for (int u = 0; u < QB; ++u)
    load_run<4 * N>(qf[u], q + ((long)b * Q + min(q0 + 16 * u + r16, Q - 1)) * ldq + (long)h * D + 4 * N * g);

  float kf[SUB][4 * N];
  auto load_k = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < SUB; ++s) load_run<4 * N>(kf[s], kb + (long)min(k0 + 16 * s + r16, K - 1) * ldk);
  };
  floatx4 o[QB][N] = {};
  float mr[QB], l[QB];
#pragma unroll
  for (int u = 0; u < QB; ++u) {
    mr[u] = NONE;
    l[u] = 0.f;
  }
  int k0 = wave * KB;
  if (k0 < K) load_k(k0);
  for (; k0 < K; k0 += WAVES * KB) {
    float vf[SUB][4][N];
    // one mask byte per lane covers the block (KB <= 64 keys); bit 16 s + 4 g + t is the lane's key (s, t)
    const uint8_t mk = mb[min(k0 + min(lane, KB - 1), K - 1)];
#pragma unroll
    for (int s = 0; s < SUB; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t) load_run<N>(vf[s][t], vb + (long)min(k0 + 16 * s + 4 * g + t, K - 1) * ldv);
    const uint64_t vis = __builtin_amdgcn_ballot_w64(mk != 0) >> (4 * g);
    floatx4 sc[QB][SUB];
#pragma unroll
    for (int u = 0; u < QB; ++u)
#pragma unroll
      for (int s = 0; s < SUB; ++s) sc[u][s] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4 * N; ++j)
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int u = 0; u < QB; ++u) sc[u][s] = mfma16_f32(kf[s][j], qf[u][j], sc[u][s]);
    if (k0 + WAVES * KB < K) load_k(k0 + WAVES * KB);
#pragma unroll
    for (int u = 0; u < QB; ++u) {
      float mx = NONE;
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float hidden = k0 + 16 * s + 4 * g + t < K ? MASK_FILL : -INFINITY;
          const float z = ((vis >> (16 * s + t)) & 1u) && hidden == MASK_FILL ? sc[u][s][t] * scale : hidden;
          sc[u][s][t] = z;
          mx = fmaxf(mx, z);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(mr[u], mx);
      const float alpha = exp_below0(mr[u] - mn);
      mr[u] = mn;
      l[u] *= alpha;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {
#pragma unroll
        for (int c = 0; c < N; ++c) o[u][c] *= alpha;
      }
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float p = exp_below0(sc[u][s][t] - mn);
          sc[u][s][t] = p;
          l[u] += p;
        }
    }
    if (k0 + KB > K) {  // keys past K count as zeros (their weight is 0, the last key's value may be infinite)
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (k0 + 16 * s + 4 * g + t >= K) {
#pragma unroll
            for (int c = 0; c < N; ++c) vf[s][t][c] = 0.f;
          }
    }
#pragma unroll
    for (int s = 0; s < SUB; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int c = 0; c < N; ++c)
#pragma unroll
          for (int u = 0; u < QB; ++u) o[u][c] = mfma16_f32(vf[s][t][c], sc[u][s][t], o[u][c]);
  }
#pragma unroll
  for (int u = 0; u < QB; ++u) {
    l[u] += __shfl_xor(l[u], 16, 64);
    l[u] += __shfl_xor(l[u], 32, 64);
    if (g == 0) {
      ms[wave][16 * u + r16] = mr[u];
      ls[wave][16 * u + r16] = l[u];
    }
    // block c, register t is dim N (4 g + t) + c of query r16
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int c = 0; c < N; ++c) os[wave][16 * u + r16][N * (4 * g + t) + c] = o[u][c][t];
  }
  __syncthreads();
  for (int idx = tid; idx < 16 * QB * D; idx += 64 * WAVES) {
    const int qi = idx / D, d = idx % D;
    if (q0 + qi >= Q) continue;
    float mx = ms[0][qi];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) mx = fmaxf(mx, ms[w][qi]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = exp_below0(ms[w][qi] - mx);
      num += os[w][qi][d] * f;
      den += ls[w][qi] * f;
    }
    out[((long)b * Q + q0 + qi) * ldo + (long)h * D + d] = num / den;
  }
}

// y[b * I + i, :] = (acc ? y : 0) + x[b * R + idx[b * I + i], :]
__global__ void __launch_bounds__(THREADS)
gather_rows_f32_kernel(const float *__restrict__ x, const int32_t *__restrict__ idx, float *__restrict__ y, int R,
                       int I, int d, long ldx, long ldy, int acc) {
  const int bi = blockIdx.x, b = bi / I;
  const int r = min(max(idx[bi], 0), R - 1);
  const float *src = x + ((long)b * R + r) * ldx;
  float *dst = y + (long)bi * ldy;
  for (int i = threadIdx.x; i < d; i += THREADS) dst[i] = acc ? dst[i] + src[i] : src[i];
}

// logits[o] = options[b, o] . base[b, qi] / sqrt(W) over the options question qi owns (owner == qi and option_mask),
// MASK_FILL elsewhere; routing = softmax over o; summary[b, qi] = sum_o routing[o] * options[b, o] (head.py:76-85).
// A workgroup takes FG questions of b and 256 columns of the summary, so the options are read once per FG questions
// there. Its waves share out the dot products of the owned options (the others need none), which every column
// block repeats: they are few next to the sum's rows.
template <int FG>
__global__ void __launch_bounds__(THREADS)
routing_f32_kernel(const float *__restrict__ options, const float *__restrict__ base, const int32_t *__restrict__ owner,
                   const uint8_t *__restrict__ option_mask, float *__restrict__ summary, int O, int NQ, int W) {
  extern __shared__ __attribute__((aligned(16))) float p[];  // [O][FG] routing weights
  constexpr int WAVES = THREADS / 64;
  const int groups = (NQ + FG - 1) / FG, b = blockIdx.x / groups, f0 = blockIdx.x % groups * FG, nf = min(FG, NQ - f0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float *ob = options + (long)b * O * W;
  const float inv = 1.0f / sqrtf((float)W);
  for (int i = threadIdx.x; i < O * FG; i += THREADS) p[i] = MASK_FILL;
  __syncthreads();
  int seen = 0;
  for (int o0 = 0; o0 < O; o0 += 64) {
    const int o = o0 + lane;
    int rel = -1;
    if (o < O && option_mask[(long)b * O + o]) rel = owner[(long)b * O + o] - f0;
    for (uint64_t bits = __builtin_amdgcn_ballot_w64(rel >= 0 && rel < nf); bits; bits &= bits - 1) {
      if (seen++ % WAVES != wave) continue;
      const int j = __builtin_ctzll(bits), f = __builtin_amdgcn_readlane(rel, j);
      const float *orow = ob + (long)(o0 + j) * W, *br = base + ((long)b * NQ + f0 + f) * W;
      float s = 0.f;
#pragma unroll 8
      for (int i = lane; i < W; i += 64) s = fmaf(orow[i], br[i], s);
      s = wave_reduce_sum(s);
      if (lane == 0) p[(o0 + j) * FG + f] = s * inv;
    }
  }
  __syncthreads();
  for (int f = wave; f < nf; f += WAVES) {
    float mx = MASK_FILL;
    for (int o = lane; o < O; o += 64) mx = fmaxf(mx, p[o * FG + f]);
    mx = wave_reduce_max(mx);
    float sum = 0.f;
    for (int o = lane; o < O; o += 64) {
      const float e = expf(p[o * FG + f] - mx);
      p[o * FG + f] = e;
      sum += e;
    }
    sum = wave_reduce_sum(sum);
    for (int o = lane; o < O; o += 64) p[o * FG + f] /= sum;
  }
  __syncthreads();
  const int i = blockIdx.y * THREADS + threadIdx.x;
  if (i >= W) return;
  float s[FG] = {};
  int o = 0;
  for (; o + 16 <= O; o += 16) {
    float v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = ob[(long)(o + e) * W + i];
#pragma unroll
    for (int e = 0; e < 16; ++e)
#pragma unroll
      for (int f = 0; f < FG; ++f) s[f] += p[(o + e) * FG + f] * v[e];
  }
  for (; o < O; ++o) {
    const float v = ob[(long)o * W + i];
#pragma unroll
    for (int f = 0; f < FG; ++f) s[f] += p[o * FG + f] * v;
  }
#pragma unroll
  for (int f = 0; f < FG; ++f)
    if (f < nf) summary[((long)b * NQ + f0 + f) * W + i] = s[f];
}

// fields[b, qi] = base[b, qi] + summary_norm[b, qi] + glob[b] + type_emb[types[b, qi]]
__global__ void __launch_bounds__(THREADS)
fields_init_f32_kernel(const float *__restrict__ base, const float *__restrict__ sn, const float *__restrict__ glob,
                       const float *__restrict__ type_emb, const int32_t *__restrict__ types, float *__restrict__ fields,
                       int NQ, int W, int num_types) {
  const int bq = blockIdx.x, b = bq / NQ;
  const int t = min(max(types[bq], 0), num_types - 1);
  for (int i = threadIdx.x; i < W; i += THREADS)
    fields[(long)bq * W + i] = ((base[(long)bq * W + i] + sn[(long)bq * W + i]) + glob[(long)b * W + i]) +
                               type_emb[(long)t * W + i];
}

DX_DEVICE float inv_length(float sumsq, float eps) { return 1.0f / fmaxf(sqrtf(sumsq), eps); }

// One workgroup per (b, o) (head.py:97-106): anchor = normalize(questions[b, owner] + glob[b]),
// prior = normalize(lexical[b, o]) . anchor * prior_scale, cosine of normalize(fields, 1e-8) and
// normalize(opts, 1e-8), features = [f, o, f * o, |f - o|]. questions / glob / lexical have H
// columns, fields / opts W.
__global__ void __launch_bounds__(THREADS)
features_f32_kernel(const float *__restrict__ fields, const float *__restrict__ opts, const float *__restrict__ questions,
                    const float *__restrict__ glob, const float *__restrict__ lexical, const int32_t *__restrict__ owner,
                    float *__restrict__ features, float *__restrict__ prior, float *__restrict__ cosine, int O, int NQ,
                    int W, int Hd, float prior_scale) {
  __shared__ float red[4][THREADS / 64];
  const int bo = blockIdx.x, b = bo / O;
  const int qi = min(max(owner[bo], 0), NQ - 1);
  const float *qr = questions + ((long)b * NQ + qi) * Hd, *gr = glob + (long)b * Hd, *lr = lexical + (long)bo * Hd;
  const float *fr = fields + (long)bo * W, *orow = opts + (long)bo * W;
  // Two passes with one reduction each (one value at a time they took six, 11.6 us for 23 options): the lengths, then
  // the two products with the features.
  float len[4] = {0.f, 0.f, 0.f, 0.f};  // of the anchor, the label vector, the field and the option
#pragma unroll 4
  for (int i = threadIdx.x; i < Hd; i += THREADS) {
    const float a = qr[i] + gr[i], l = lr[i];
    len[0] += a * a;
    len[1] += l * l;
  }
#pragma unroll 4
  for (int i = threadIdx.x; i < W; i += THREADS) {
    const float f = fr[i], o = orow[i];
    len[2] += f * f;
    len[3] += o * o;
  }
  block_sums(len, red);
  const float ia = inv_length(len[0], 1e-12f), il = inv_length(len[1], 1e-12f);
  const float jf = inv_length(len[2], 1e-8f), jo = inv_length(len[3], 1e-8f);
  float dots[2] = {0.f, 0.f};
#pragma unroll 4
  for (int i = threadIdx.x; i < Hd; i += THREADS) dots[0] += (lr[i] * il) * ((qr[i] + gr[i]) * ia);
  float *ft = features + (long)bo * 4 * W;
#pragma unroll 4
  for (int i = threadIdx.x; i < W; i += THREADS) {
    const float f = fr[i], o = orow[i];
    dots[1] += (f * jf) * (o * jo);
    ft[i] = f;
    ft[W + i] = o;
    ft[2 * W + i] = f * o;
    ft[3 * W + i] = fabsf(f - o);
  }
  block_sums(dots, red);
  const float dp = dots[0], cs = dots[1];
  if (threadIdx.x == 0) {
    prior[bo] = dp * prior_scale;
    cosine[bo] = cs;
  }
}

// out[b, o] = option_mask ? prior + gate * (joint_scale * cosine + residual) : -1e9
__global__ void __launch_bounds__(THREADS)
combine_f32_kernel(const float *__restrict__ prior, const float *__restrict__ cosine, const float *__restrict__ residual,
                   const uint8_t *__restrict__ option_mask, float *__restrict__ out, long n, float gate,
                   float joint_scale) {
  const long i = (long)blockIdx.x * THREADS + threadIdx.x;
  if (i >= n) return;
  out[i] = option_mask[i] ? prior[i] + gate * (joint_scale * cosine[i] + residual[i]) : -1e9f;
}

// The same with the learned scalars still on the device: out = prior_scale prior + gate (joint_scale cosine +
// residual), scales exp(min(s, ln 100)) and gate sigmoid(g), each rounded once from double. Asking the host for them
// stalled the forward three times.
__global__ void __launch_bounds__(THREADS)
combine_scaled_f32_kernel(const float *__restrict__ prior, const float *__restrict__ cosine,
                          const float *__restrict__ residual, const uint8_t *__restrict__ option_mask,
                          const float *__restrict__ prior_logit_scale, const float *__restrict__ joint_logit_scale,
                          const float *__restrict__ residual_gate, float *__restrict__ out, long n) {
  const long i = (long)blockIdx.x * THREADS + threadIdx.x;
  if (i >= n) return;
  auto scale = [](float v) {
    const double most = 4.605170185988092;  // ln 100
    return (float)exp((double)v > most ? most : (double)v);
  };
  const float ps = scale(*prior_logit_scale), js = scale(*joint_logit_scale);
  const float gate = (float)(1.0 / (1.0 + exp(-(double)*residual_gate)));
  out[i] = option_mask[i] ? ps * prior[i] + gate * (js * cosine[i] + residual[i]) : -1e9f;
}

unsigned blocks(long n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

hipError_t dx_layer_norm_f32_launch(const float *x, const float *w, const float *b, float *y, long rows, int d,
                                    long ldx, long ldy, float eps, hipStream_t s) {
  const uintptr_t addr = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) |
                         reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(y);
  const unsigned grid = blocks(rows, THREADS / 64);
  if (d % 4 == 0 && d <= 4096 && ((ldx | ldy) & 3) == 0 && (addr & 15) == 0) {
    auto kern = d <= 1024 ? layer_norm_f32_row_kernel<4> : layer_norm_f32_row_kernel<16>;
    kern<<<grid, THREADS, 0, s>>>(x, w, b, y, rows, d, ldx, ldy, eps);
    return hipGetLastError();
  }
  layer_norm_f32_kernel<<<grid, THREADS, 0, s>>>(x, w, b, y, rows, d, ldx, ldy, eps);
  return hipGetLastError();
}

template <int TM, int TN>
static void linear_run(const float *x, const float *w, const float *bias, float *y, long m, int n, int k, long ldx,
                       long ldw, long ldy, int act, int acc, hipStream_t s) {
  const bool vec = ((ldx | ldw) & 3) == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) == 0;
  auto kern = vec ? linear_f32_kernel<TM, TN, true> : linear_f32_kernel<TM, TN, false>;
  kern<<<blocks(n, 16 * TN) * blocks(m, 16 * TM), 256, 0, s>>>(x, w, bias, y, m, n, k, ldx, ldw, ldy, act, acc);
}

hipError_t dx_linear_f32_launch(const float *x, const float *w, const float *bias, float *y, long m, int n, int k,
                                long ldx, long ldw, long ldy, int act, int acc, hipStream_t s) {
  // n, k, strides and alignment choose between the split products and the fp32 ones (another order of the sums); m, by
  // the rounds of tiles over the chip, only a tile shape.
  auto tiles = [&](int tm, int tn) { return (m + tm - 1) / tm * ((n + tn - 1) / tn); };
  // the split kernels read whole 16-byte chunks of a row through 32-bit offsets
  const bool chunks = k >= 64 && ((k | ldx | ldw) & 3) == 0 && ldx <= (1 << 20) && ldw <= (1 << 20) &&
                      ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) == 0;
  if (chunks) {
    const int vec_y = (ldy & 3) == 0 && ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(bias)) & 15) == 0;
    // us per 1024 k: 128 x 128 tiles 46 a round of 256 workgroups and 17, 128 x 64 tiles 28 and 6, 32 x 32 tiles 7 for
    // one round, then 2 and 0.0215 a tile. Measured us, 32 x 32 / 128 x 64 / 128 x 128 (fp32 or split products chosen by
    // m, before):
    //   23 x 1024 x 1024: 8 / 33 / 56 (6)       23 x 1024 x 4096: 22 / 126 / 210 (20)     200 x 1024 x 4096: 24 / 137 / 212 (34)
    //   600 x 1024 x 4096: 67 / 139 / 214 (73)  600 x 2048 x 1024: 29 / 38 / 59 (35)      2000 x 1024 x 1024: 45 / 42 / 61 (38)
    //   4096 x 1024 x 1024: 89 / 63 / 69 (59)   4096 x 1024 x 4096: 339 / 229 / 231 (197)
    //   4096 x 2048 x 4096: 689 / 453 / 374 (357)
    //   32768 x 1024 x 4096: 2812 / 1619 / 1395 (1296)
    const long wide = tiles(128, 128), slim = tiles(128, 64), few = tiles(32, 32);
    const double wide_us = 46. * ((wide + 255) / 256) + 17, slim_us = 28. * ((slim + 255) / 256) + 6;
    const double few_us = few <= 256 ? 7 : 0.0215 * few + 2;
    if (few_us <= fmin(wide_us, slim_us)) {
      // eight parts of k at once, or four in rings of 32 columns
      if (k <= 4 * PART)
        linear_split_small_kernel<4, 32, 2><<<(unsigned)few, 256, 0, s>>>(x, w, bias, y, m, n, k, ldx, ldw, ldy, act, acc,
                                                                         vec_y);
      else
        linear_split_small_kernel<8, 16, 2><<<(unsigned)few, 512, 0, s>>>(x, w, bias, y, m, n, k, ldx, ldw, ldy, act, acc,
                                                                         vec_y);
    } else if (wide_us <= slim_us) {
      linear_split_kernel<2, 2><<<(unsigned)wide, 256, 0, s>>>(x, w, bias, y, m, n, k, ldx, ldw, ldy, act, acc, vec_y);
    } else {
      linear_split_kernel<2, 1><<<(unsigned)slim, 256, 0, s>>>(x, w, bias, y, m, n, k, ldx, ldw, ldy, act, acc, vec_y);
    }
    return hipGetLastError();
  }
  // A tile's time is its rounds of waves over the 1024 SIMDs times a wave's share of one 64 x 64 x k product; a 64 x 32
  // or 32 x 32 wave, which re-reads its operands more often, runs at 0.7 or 0.55 of the 64 x 64 wave's rate.
  auto rounds = [](long waves) { return (double)((waves + 1023) / 1024); };
  const double cost[3] = {rounds(4 * tiles(64, 64)) / 4, rounds(4 * tiles(64, 32)) / 8 * 1.45,
                          rounds(4 * tiles(32, 32)) / 16 * 1.8};
  if (cost[0] <= fmin(cost[1], cost[2])) linear_run<4, 4>(x, w, bias, y, m, n, k, ldx, ldw, ldy, act, acc, s);
  else if (cost[1] <= cost[2]) linear_run<4, 2>(x, w, bias, y, m, n, k, ldx, ldw, ldy, act, acc, s);
  else linear_run<2, 2>(x, w, bias, y, m, n, k, ldx, ldw, ldy, act, acc, s);
  return hipGetLastError();
}

hipError_t dx_span_means_f32_launch(const float *x, const int32_t *spans, float *out, int B, int S, int O, int d,
                                    long ldx, long ldo, hipStream_t s) {
  span_means_f32_kernel<false><<<dim3((unsigned)(B * O), blocks(d, THREADS)), THREADS, 0, s>>>(x, nullptr, spans, out, 0,
                                                                                             S, O, d, ldx, ldo);
  return hipGetLastError();
}

hipError_t dx_span_means_gather_f32_launch(const float *x, const int32_t *index, const int32_t *spans, float *out, int B,
                                           int R, int S, int O, int d, long ldx, long ldo, hipStream_t s) {
  span_means_f32_kernel<true><<<dim3((unsigned)(B * O), blocks(d, THREADS)), THREADS, 0, s>>>(x, index, spans, out, R, S,
                                                                                            O, d, ldx, ldo);
  return hipGetLastError();
}

template <int N>
static void mha_run(const float *q, const float *k, const float *v, const uint8_t *key_mask, float *out, int B, int Q,
                    int K, int H, long ldq, long ldk, long ldv, long ldo, hipStream_t s) {
  // Eight waves and SUB blocks of 16 keys a step (as many as leave registers for two waves per SIMD, the softmax of one
  // beside the products of the other) at every size, so that a row's sums do not depend on the launch; its size picks
  // 16 or 32 queries alone. us, 4 waves -> 8, 16 heads x 64: 1 x 23 x 600 11.9 -> 11.8, 8 x 64 x 4096 169 -> 164,
  // 8 x 512 x 4096 657 -> 677; 8 heads x 128, 2 x 100 x 1500 48 -> 47. SUB 4 at head_dim 64: 14, 163 and 860.
  constexpr int SUB = N <= 2 ? 4 : N <= 5 ? 2 : 1;
  if ((long)B * H * ((Q + 31) / 32) >= 512)
    mha_f32_mfma_kernel<N, 2, 8, SUB><<<dim3((Q + 31) / 32, H, B), 512, 0, s>>>(q, k, v, key_mask, out, Q, K, ldq, ldk,
                                                                             ldv, ldo);
  else
    mha_f32_mfma_kernel<N, 1, 8, SUB><<<dim3((Q + 15) / 16, H, B), 512, 0, s>>>(q, k, v, key_mask, out, Q, K, ldq, ldk,
                                                                             ldv, ldo);
}

hipError_t dx_mha_f32_launch(const float *q, const float *k, const float *v, const uint8_t *key_mask, float *out,
                             int B, int Q, int K, int H, int dh, long ldq, long ldk, long ldv, long ldo, hipStream_t s) {
  const uintptr_t addr = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v);
  if (dh % 16 == 0 && dh <= 128 && ((ldq | ldk | ldv) & 3) == 0 && (addr & 15) == 0 && H <= 65535 && B <= 65535) {
    switch (dh / 16) {
      case 1: mha_run<1>(q, k, v, key_mask, out, B, Q, K, H, ldq, ldk, ldv, ldo, s); break;
      case 2: mha_run<2>(q, k, v, key_mask, out, B, Q, K, H, ldq, ldk, ldv, ldo, s); break;
      case 3: mha_run<3>(q, k, v, key_mask, out, B, Q, K, H, ldq, ldk, ldv, ldo, s); break;
      case 4: mha_run<4>(q, k, v, key_mask, out, B, Q, K, H, ldq, ldk, ldv, ldo, s); break;
      case 5: mha_run<5>(q, k, v, key_mask, out, B, Q, K, H, ldq, ldk, ldv, ldo, s); break;
      case 6: mha_run<6>(q, k, v, key_mask, out, B, Q, K, H, ldq, ldk, ldv, ldo, s); break;
      case 7: mha_run<7>(q, k, v, key_mask, out, B, Q, K, H, ldq, ldk, ldv, ldo, s); break;
      default: mha_run<8>(q, k, v, key_mask, out, B, Q, K, H, ldq, ldk, ldv, ldo, s); break;
    }
    return hipGetLastError();
  }
  const size_t shm = ((size_t)K + THREADS) * sizeof(float);
  mha_f32_kernel<<<(unsigned)(B * Q * H), THREADS, shm, s>>>(q, k, v, key_mask, out, Q, K, H, dh, ldq, ldk, ldv, ldo);
  return hipGetLastError();
}

hipError_t dx_gather_rows_f32_launch(const float *x, const int32_t *idx, float *y, int B, int R, int I, int d,
                                     long ldx, long ldy, int acc, hipStream_t s) {
  gather_rows_f32_kernel<<<(unsigned)(B * I), THREADS, 0, s>>>(x, idx, y, R, I, d, ldx, ldy, acc);
  return hipGetLastError();
}

hipError_t dx_routing_f32_launch(const float *options, const float *base, const int32_t *owner,
                                 const uint8_t *option_mask, float *summary, int B, int O, int NQ, int W,
                                 hipStream_t s) {
  // eight questions per workgroup where that still fills the chip and their weights fit 64 KB of LDS
  const unsigned cols = blocks(W, THREADS);
  if (O <= 2048 && (long)B * blocks(NQ, 8) * cols >= 128)
    routing_f32_kernel<8><<<dim3(B * blocks(NQ, 8), cols), THREADS, (size_t)O * 8 * sizeof(float), s>>>(
        options, base, owner, option_mask, summary, O, NQ, W);
  else
    routing_f32_kernel<1><<<dim3((unsigned)(B * NQ), cols), THREADS, (size_t)O * sizeof(float), s>>>(options, base, owner,
                                                                                      option_mask, summary, O, NQ, W);
  return hipGetLastError();
}

hipError_t dx_fields_init_f32_launch(const float *base, const float *sn, const float *glob, const float *type_emb,
                                     const int32_t *types, float *fields, int B, int NQ, int W, int num_types,
                                     hipStream_t s) {
  fields_init_f32_kernel<<<(unsigned)(B * NQ), THREADS, 0, s>>>(base, sn, glob, type_emb, types, fields, NQ, W,
                                                                num_types);
  return hipGetLastError();
}

hipError_t dx_features_f32_launch(const float *fields, const float *opts, const float *questions, const float *glob,
                                  const float *lexical, const int32_t *owner, float *features, float *prior,
                                  float *cosine, int B, int O, int NQ, int W, int Hd, float prior_scale,
                                  hipStream_t s) {
  features_f32_kernel<<<(unsigned)(B * O), THREADS, 0, s>>>(fields, opts, questions, glob, lexical, owner, features,
                                                            prior, cosine, O, NQ, W, Hd, prior_scale);
  return hipGetLastError();
}

hipError_t dx_combine_f32_launch(const float *prior, const float *cosine, const float *residual,
                                 const uint8_t *option_mask, float *out, long n, float gate, float joint_scale,
                                 hipStream_t s) {
  combine_f32_kernel<<<blocks(n, THREADS), THREADS, 0, s>>>(prior, cosine, residual, option_mask, out, n, gate,
                                                            joint_scale);
  return hipGetLastError();
}

hipError_t dx_combine_scaled_f32_launch(const float *prior, const float *cosine, const float *residual,
                                        const uint8_t *option_mask, const float *prior_logit_scale,
                                        const float *joint_logit_scale, const float *residual_gate, float *out, long n,
                                        hipStream_t s) {
  combine_scaled_f32_kernel<<<blocks(n, THREADS), THREADS, 0, s>>>(prior, cosine, residual, option_mask,
                                                                  prior_logit_scale, joint_logit_scale, residual_gate,
                                                                  out, n);
  return hipGetLastError();
}
