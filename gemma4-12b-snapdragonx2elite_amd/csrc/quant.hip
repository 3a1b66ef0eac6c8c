// Weight preparation on the GPU (load time): the int4 block quantizer, the
// e4m3 scale lift, the W8A8 int8 fold, the W4A8 ratio and the repacks from
// the reference engine's storage layouts into the panel-64 device layout.
//
// Arithmetic follows the reference quantizer quant() (src/vk_engine.py:125-159)
// operation for operation: IEEE fp32 divides (__fdiv_rn), products rounded
// once (__fmul_rn), round-half-to-even (rintf), RNE narrowing to fp16. The
// outputs are bit-identical to the numpy quantizer.
#include "q4mi_common.h"

namespace q4 {

// ---- int4 block quantizer (src/vk_engine.py:126-131) ---------------------
// A workgroup quantizes 64 rows (one panel) x QB blocks; each wave takes 16
// rows, 8 / QB rows' blocks (1 KB) per load, all 2 QB loads requested before
// the first is used: 8 lanes hold a block, 4 consecutive elements each, the
// block's maximum is an 8-lane reduction, and lane pairs join their nibbles
// to device words. Units and fp16 scales go through LDS to the panel order
// (64 rows of a block contiguous), fp32 scales are stored from the lanes.
// Bound by the read of W: 15360 x 3840 (236 MB in, 41 MB out) 73.4 -> 63.2 us
// against a thread per block, whose 16-byte loads of a wave lay 64 rows apart.
// QB = 4 reads whole 512-byte runs of a row; with QB = 1 four times the
// workgroups run a quarter of the chain each, better up to QUANT_SMALL values
// (QB 4 / 1 / a thread per block, W not in cache: 64 x 3840 5.8 / 4.3 / 5.1 us, 1000
// x 3840 8.5 / 7.1 / 7.3, 4000 x 3840 21.1 / 21.0 / 22.0, 8000 x 3840 34.6 / 38.4 /
// 40.0).
// The code is rint(v / sc) of the correctly rounded quotient; v times the
// approximate reciprocal differs from it by less than 2e-6 (|v / sc| <= 7,
// three roundings and the 1-ulp reciprocal), so only values that close to a
// rounding tie, or not finite, take the division.
constexpr long QUANT_SMALL = 24L << 20;
template <int QB>
__global__ void __launch_bounds__(256) quantize_kernel(const float* __restrict__ W, int N, int K, int nblk,
                                                       uint4* __restrict__ wq, uint16_t* __restrict__ sc16,
                                                       float* __restrict__ sc32) {
  constexpr int LPR = 8 * QB, RL = 64 / LPR, NL = 16 / RL;  // lanes per row, rows per load, loads per wave
  __shared__ __attribute__((aligned(16))) uint32_t words[PANEL][QB * 4 + 4];
  __shared__ uint16_t scs[QB][PANEL];
  const int ct = ceil_div(nblk, QB);
  const int p = blockIdx.x / ct, b0 = (blockIdx.x % ct) * QB;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane / LPR, lc = lane % LPR, lb = lc >> 3;  // the lane's row of a load, place in the row, block
  const int b = b0 + lb;
  const bool bok = b < nblk;
  float4 v[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int n = p * PANEL + wave * 16 + i * RL + lr;
    v[i] = bok && n < N ? *reinterpret_cast<const float4*>(W + (long)n * K + (long)b0 * BLK + 4 * lc)
                        : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  // nibble shifts of this lane's elements e = 4 (lane & 1) + c of its word
  const int odd = lane & 1;
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int r = wave * 16 + i * RL + lr, n = p * PANEL + r;
    const float x[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
    const float amax = reduce8<true>(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))));
    const float sc = fmaxf(__fdiv_rn(amax, 7.0f), 1e-8f);
    const float inv = __builtin_amdgcn_rcpf(sc);
    float c[4];
    bool near = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float t = x[e] * inv;
      c[e] = rintf(t);
      near |= !(fabsf(t - c[e]) < 0.499996f);
    }
    if (near) {
#pragma unroll
      for (int e = 0; e < 4; ++e) c[e] = rintf(__fdiv_rn(x[e], sc));
    }
    uint32_t w = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w |= ((uint32_t)fminf(fmaxf(c[e] + 8.0f, 0.0f), 15.0f) & 15u) << (4 * nib_pos(e));
    w <<= 8 * odd;   // elements 4..7 sit two nibbles above 0..3
    w |= __float_as_uint(dpp_f<DPP_XOR1>(__uint_as_float(w)));
    const bool live = n < N;
    if (!odd) words[r][lc >> 1] = live ? w : 0x88888888u;   // padded row: code 8 (= weight 0), scale 0
    if ((lane & 7) == 0) {
      scs[lb][r] = live ? f2h_after_f32(sc) : (uint16_t)0;
      if (sc32 && live && bok) sc32[(long)n * nblk + b] = sc;
    }
  }
  __syncthreads();
#pragma unroll
  for (int bb = wave; bb < QB; bb += 4) {
    if (b0 + bb >= nblk) break;
    const long u = ((long)p * nblk + b0 + bb) * PANEL + lane;
    wq[u] = *reinterpret_cast<const uint4*>(&words[lane][4 * bb]);
    sc16[u] = scs[bb][lane];
  }
}

// ---- e4m3 scale lift (src/vk_engine.py:133-137) ---------------------------
__global__ void zero_word_kernel(uint32_t* __restrict__ p) { *p = 0u; }

// One atomic per workgroup and 256 workgroups of 1024 threads: atomics on one
// address are served one after the other, and one per wave of 4096 waves was
// most of the kernel's time (7.4 MB: 49.2 -> 5.3 us).
__global__ void __launch_bounds__(1024) absmax_bits_kernel(const float* __restrict__ x, long n,
                                                           uint32_t* __restrict__ out) {
  __shared__ float red[16];
  float m = 0.0f;
  const long stride = (long)gridDim.x * 1024;
  long i = (long)blockIdx.x * 1024 + threadIdx.x;
  for (; i + 3 * stride < n; i += 4 * stride)  // four independent loads in flight
    m = fmaxf(m, fmaxf(fmaxf(fabsf(x[i]), fabsf(x[i + stride])), fmaxf(fabsf(x[i + 2 * stride]), fabsf(x[i + 3 * stride]))));
  for (; i < n; i += stride) m = fmaxf(m, fabsf(x[i]));
  m = reduce64<true>(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x < 64) {
    m = reduce16<true>(red[threadIdx.x & 15]);
    if (threadIdx.x == 0) atomicMax(out, __float_as_uint(m));  // m >= 0: bit order == value order
  }
}

// float32 in [0, 448] -> e4m3fn byte, round-half-to-even. Normal band:
// round the fp32 bit pattern at mantissa bit 20 (keeping 3 mantissa bits)
// and rebias the exponent from 127 to 7; a rounding carry moves into the
// exponent by itself. Subnormal band (< 2^-6): the value in units of 2^-9,
// rounded to even (code 8 is the smallest normal, 2^-6).
__device__ inline uint32_t e4m3_encode_pos(float v) {
  if (v < 0.015625f) return (uint32_t)rintf(v * 512.0f);
  uint32_t bits = __float_as_uint(v);
  uint32_t r = (bits + 0x7FFFFu + ((bits >> 20) & 1u)) >> 20;
  return r - (120u << 3);
}

__device__ inline int lift_shift(const uint32_t* maxbits) {
  float mx = __uint_as_float(*maxbits);
  if (!(mx > 0.0f)) return 0;
  int e;
  frexp(256.0 / (double)mx, &e);  // 256/mx = f * 2^e, f in [0.5, 1): floor(log2) = e - 1
  return e - 1;
}

// A workgroup lifts 64 rows (one panel) x 32 blocks: rows are read along the
// blocks (128 bytes per row) and stored in panel order through LDS (15360 x
// 120 scales: 11.5 -> 4.2 us against lanes along the rows).
__global__ void __launch_bounds__(256) e4m3_lift_kernel(const float* __restrict__ sc32, int N, int nblk,
                                                        const uint32_t* __restrict__ maxbits,
                                                        uint8_t* __restrict__ sc8, float* __restrict__ inv_out) {
  constexpr int TB = 32;
  __shared__ __attribute__((aligned(4))) uint8_t out[TB][PANEL + 4];
  const int ct = ceil_div(nblk, TB);
  const int p = blockIdx.x / ct, b0 = (blockIdx.x % ct) * TB;
  const int c = threadIdx.x & (TB - 1), r0 = threadIdx.x / TB;
  float x[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int n = p * PANEL + 8 * i + r0;
    x[i] = n < N && b0 + c < nblk ? sc32[(long)n * nblk + b0 + c] : 0.0f;  // padded rows: scale 0
  }
  const int shift = lift_shift(maxbits);
  if (blockIdx.x == 0 && threadIdx.x == 0 && inv_out) *inv_out = ldexpf(1.0f, -shift);
  const float p2 = __int_as_float((shift + 127) << 23);  // 2^shift, exact
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int n = p * PANEL + 8 * i + r0;
    const float v = fminf(fmaxf(__fmul_rn(x[i], p2), 0.0f), 448.0f);
    out[c][8 * i + r0] = n < N ? (uint8_t)e4m3_encode_pos(v) : (uint8_t)0;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < TB * 16; i += 256) {
    const int bb = i >> 4, w = i & 15;
    if (b0 + bb < nblk)  // one 4-byte store, at any alignment of sc8
      __builtin_memcpy(sc8 + ((long)p * nblk + b0 + bb) * PANEL + 4 * w, &out[bb][4 * w], 4);
  }
}

// ---- W8A8 fold (src/vk_engine.py:152-157) --------------------------------
// A workgroup folds FR rows: thread (r = t % FR, block t / FR + 256 / FR i). With
// FR = 8 the 8 rows of a block are one 128-byte line of units, read by one
// workgroup (a workgroup per row fetched every line into the L2 of all 8
// XCDs). The row maximum needs only the block's largest |code| (products
// round monotonically). The 32 quotients of a block take 9 values: k s for k =
// 0..8 with either sign, so a thread rounds 8 quotients, packs the 16 codes'
// bytes into 4 words and looks the codes up with byte permutes. W8 is row-major
// [N][K] or, PACKED, the layout of the packed W8A8 GEMM (1 KB per 32 rows x
// 32 k: 16-byte chunk l is row l % 32, k half l / 32; rows padded to 32 and
// K to 128 with zeros), which saves the pass that packs it.
// 15360 x 3840: 59.6 us for the row-major fold and 18.3 for its packing
// before, 24.1 us in one pass (96 MB). Below FOLD_ROWS rows 8-row workgroups
// do not fill the chip and each is a long chain of rounds: FR = 2 (8 / 2, and a
// workgroup per row: 8 x 3840 6.4 / 4.3 / 4.8 us, 300 x 15360 18.9 / 7.7 / 11.3, 1000 x
// 3840 7.1 / 5.8 / 9.4, 1000 x 15360 20.0 / 13.0 / 26.5, 2000 x 3840 7.9 / 7.5 / 13.2,
// packed 7.5 / 8.7).
constexpr int FOLD_ROWS = 1536;
__device__ inline uint32_t fold_byte(float v) {
  return (uint32_t)(int)fminf(fmaxf(v, -127.0f), 127.0f) & 0xFFu;
}
// bytes of the 4 codes in the low nibbles of c's bytes; t: the 16 codes' bytes
__device__ inline uint32_t fold_lookup(uint32_t c, const uint32_t (&t)[4]) {
  const uint32_t lo = __builtin_amdgcn_perm(t[1], t[0], c & 0x07070707u);
  const uint32_t hi = __builtin_amdgcn_perm(t[3], t[2], c & 0x07070707u);
  return __builtin_amdgcn_perm(hi, lo, ((c >> 1) & 0x04040404u) | 0x03020100u);  // byte i of hi where bit 3 is set
}

template <bool PACKED, int FR>
__global__ void __launch_bounds__(256) w8_fold_kernel(const uint4* __restrict__ wq, const float* __restrict__ sc32,
                                                      int N, int K, int nblk, int8_t* __restrict__ W8,
                                                      float* __restrict__ sw32, uint16_t* __restrict__ sw16,
                                                      int kslices) {
  constexpr int FB = 256 / FR;
  __shared__ float red[4][FR];
  const int r = threadIdx.x & (FR - 1), n = blockIdx.x * FR + r, bt = threadIdx.x / FR;
  const bool live = n < N;
  const long u0 = panel_index(n < N ? n : N - 1, 0, nblk);
  const float* srow = sc32 + (long)(live ? n : N - 1) * nblk;
  float amax = 0.0f;
  for (int b = bt; b < nblk; b += FB) {
    const uint4 w = wq[u0 + (long)b * PANEL];
    const float s = srow[b];
    typedef unsigned short v2us __attribute__((ext_vector_type(2)));
    v2us mx = {8, 8}, mn = {8, 8};  // the block's largest and smallest code (and 8 = weight 0)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t wi = i == 0 ? w.x : i == 1 ? w.y : i == 2 ? w.z : w.w;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const v2us c = __builtin_bit_cast(v2us, (wi >> (4 * k)) & 0x000F000Fu);
        mx = __builtin_elementwise_max(mx, c);
        mn = __builtin_elementwise_min(mn, c);
      }
    }
    const int far = max(max((int)mx.x, (int)mx.y) - 8, 8 - min((int)mn.x, (int)mn.y));
    amax = fmaxf(amax, fabsf(__fmul_rn((float)far, s)));
  }
  amax = slot_reduce<FR, true>(amax);
  if ((threadIdx.x & 63) < FR) red[threadIdx.x >> 6][r] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0][r], red[1][r]), fmaxf(red[2][r], red[3][r]));
  const float sw = fmaxf(__fdiv_rn(amax, 127.0f), 1e-12f);
  if (threadIdx.x < FR && live) {
    if (sw32) sw32[n] = sw;
    if (sw16) sw16[n] = f2h_after_f32(sw);
  }
  if (!PACKED && !live) return;
  const int nb_out = PACKED ? kslices : nblk;
  for (int b = bt; b < nb_out; b += FB) {
    uint32_t o[8] = {};
    if (live && b < nblk) {
      const uint4 wv = wq[u0 + (long)b * PANEL];
      const float s = srow[b];
      uint32_t t[4];
      uint32_t pos[9], neg[9];
      pos[0] = fold_byte(__fmul_rn(0.0f, s));  // 0, or -127 for a scale that is not finite
#pragma unroll
      for (int k = 1; k <= 8; ++k) {
        const float v = rintf(__fdiv_rn(__fmul_rn((float)k, s), sw));
        pos[k] = fold_byte(v);
        neg[k] = fold_byte(-v);
      }
      t[0] = neg[8] | (neg[7] << 8) | (neg[6] << 16) | (neg[5] << 24);
      t[1] = neg[4] | (neg[3] << 8) | (neg[2] << 16) | (neg[1] << 24);
      t[2] = pos[0] | (pos[1] << 8) | (pos[2] << 16) | (pos[3] << 24);
      t[3] = pos[4] | (pos[5] << 8) | (pos[6] << 16) | (pos[7] << 24);
      const uint32_t w[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // low nibbles hold elements 0, 4, 1, 5 and high nibbles 2, 6, 3, 7 of the word
        const uint32_t lo = fold_lookup(w[i] & 0x0F0F0F0Fu, t), hi = fold_lookup((w[i] >> 4) & 0x0F0F0F0Fu, t);
        o[2 * i] = __builtin_amdgcn_perm(hi, lo, 0x06040200u);
        o[2 * i + 1] = __builtin_amdgcn_perm(hi, lo, 0x07050301u);
      }
    }
    uint4* dst;
    long half;
    if constexpr (PACKED) {
      dst = reinterpret_cast<uint4*>(W8 + ((long)(n >> 5) * kslices + b) * 1024) + (n & 31);
      half = 32;
    } else {
      dst = reinterpret_cast<uint4*>(W8 + (long)n * K + (long)b * BLK);
      half = 1;
    }
    dst[0] = make_uint4(o[0], o[1], o[2], o[3]);
    dst[half] = make_uint4(o[4], o[5], o[6], o[7]);
  }
}

// ---- W4A8 ratio (benchmarks/coopgemm_w4a8.py:84) --------------------------
__global__ void w4a8_ratio_kernel(const float* __restrict__ sc32, const float* __restrict__ sw32, int N, int nblk,
                                  uint16_t* __restrict__ ratio) {
  long u = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long units = (long)pad_rows(N) * nblk;
  if (u >= units) return;
  int r = (int)(u % PANEL);
  long pb = u / PANEL;
  int b = (int)(pb % nblk);
  int n = (int)(pb / nblk) * PANEL + r;
  ratio[u] = (n < N) ? f2h_after_f32(__fdiv_rn(sc32[(long)n * nblk + b], sw32[n])) : (uint16_t)0;
}

// ---- repacks from the reference layouts ----------------------------------
__global__ void repack_ref_kernel(const uint32_t* __restrict__ wp, const uint16_t* __restrict__ sc_ref, int N, int K,
                                  int nblk, uint4* __restrict__ wq, uint16_t* __restrict__ sc_dev) {
  long u = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long units = (long)pad_rows(N) * nblk;
  if (u >= units) return;
  int r = (int)(u % PANEL);
  long pb = u / PANEL;
  int b = (int)(pb % nblk);
  int n = (int)(pb / nblk) * PANEL + r;
  if (n >= N) {
    if (wq) wq[u] = make_uint4(0x88888888u, 0x88888888u, 0x88888888u, 0x88888888u);
    if (sc_dev) sc_dev[u] = 0;
    return;
  }
  if (wq) {
    const int n8 = N / 8, shift = 4 * (n % 8);
    uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < BLK; ++k) {
      uint32_t q = (wp[(long)(b * BLK + k) * n8 + n / 8] >> shift) & 15u;
      w[k >> 3] |= q << (4 * nib_pos(k & 7));
    }
    wq[u] = make_uint4(w[0], w[1], w[2], w[3]);
  }
  if (sc_dev) sc_dev[u] = sc_ref[(long)b * N + n];
}

__global__ void repack_e4m3_ref_kernel(const uint8_t* __restrict__ sc_ref, int N, int nblk, uint8_t* __restrict__ sc_dev) {
  long u = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long units = (long)pad_rows(N) * nblk;
  if (u >= units) return;
  int r = (int)(u % PANEL);
  long pb = u / PANEL;
  int b = (int)(pb % nblk);
  int n = (int)(pb / nblk) * PANEL + r;
  sc_dev[u] = (n < N) ? sc_ref[(long)b * N + n] : (uint8_t)0;
}

__global__ void transpose_i8_kernel(const int8_t* __restrict__ src, int rows, int cols, int8_t* __restrict__ dst) {
  // src [rows][cols] -> dst [cols][rows]; 64x64 tiles through LDS.
  __shared__ int8_t tile[64][65];
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  for (int i = threadIdx.x; i < 64 * 64; i += blockDim.x) {
    int r = i / 64, c = i % 64;
    if (r0 + r < rows && c0 + c < cols) tile[r][c] = src[(long)(r0 + r) * cols + c0 + c];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * 64; i += blockDim.x) {
    int c = i / 64, r = i % 64;
    if (r0 + r < rows && c0 + c < cols) dst[(long)(c0 + c) * rows + r0 + r] = tile[r][c];
  }
}

// Two panel-64 matrices A, B (N rows each, N % 32 == 0) -> one of 2N rows
// with row 2i = A row i and row 2i + 1 = B row i, units and scales (sb
// bytes each) moved as they are. One thread per output (row, block) unit.
__global__ void interleave_rows_kernel(const uint4* __restrict__ wa, const uint8_t* __restrict__ sa,
                                       const uint4* __restrict__ wb, const uint8_t* __restrict__ sbp, int nblk,
                                       int sbytes, uint4* __restrict__ wo, uint8_t* __restrict__ so, long units) {
  const long u = (long)blockIdx.x * 256 + threadIdx.x;
  if (u >= units) return;
  const int r64 = (int)(u % PANEL);
  const long pb = u / PANEL;  // panel * nblk + block
  const int b = (int)(pb % nblk);
  const int n2 = (int)(pb / nblk) * PANEL + r64;  // output row
  const int n = n2 >> 1;
  const long src = ((long)(n / PANEL) * nblk + b) * PANEL + n % PANEL;
  const bool odd = n2 & 1;
  wo[u] = odd ? wb[src] : wa[src];
  const uint8_t* sp = (odd ? sbp : sa) + src * sbytes;
  for (int i = 0; i < sbytes; ++i) so[u * sbytes + i] = sp[i];
}

static int check_wk(int N, int K) {
  Q4_ARG(N > 0 && K > 0 && K % BLK == 0, "bad shape N=%d K=%d (K must be a positive multiple of 32)", N, K);
  Q4_ARG((long)N * K < (1L << 40), "matrix too large");
  return Q4_OK;
}

}  // namespace q4

using namespace q4;

extern "C" {

int q4_quantize(const float* W, int N, int K, uint32_t* wq, uint16_t* sc16, float* sc32, void* stream) {
  clear_error();
  if (int st = check_wk(N, K)) return st;
  Q4_ARG(W && wq && sc16, "null pointer");
  Q4_ARG(((uintptr_t)W & 15) == 0 && ((uintptr_t)wq & 15) == 0, "W and wq must be 16-byte aligned");
  const int nblk = K / BLK;
  const bool small = (long)N * K <= QUANT_SMALL;
  const long wgs = (long)(pad_rows(N) / PANEL) * (small ? nblk : ceil_div(nblk, 4));
  Q4_ARG(wgs < (1L << 31), "matrix too large");
  hipLaunchKernelGGL(small ? quantize_kernel<1> : quantize_kernel<4>, dim3((unsigned)wgs), dim3(256), 0,
                     as_stream(stream), W, N, K, nblk, reinterpret_cast<uint4*>(wq), sc16, sc32);
  Q4_LAUNCHED("quantize");
  return Q4_OK;
}

int q4_scales_e4m3(const float* sc32, int N, int K, uint8_t* sc8, float* inv_dev, uint32_t* work, void* stream) {
  clear_error();
  if (int st = check_wk(N, K)) return st;
  Q4_ARG(sc32 && sc8 && work, "null pointer");
  const int nblk = K / BLK;
  long n = (long)N * nblk;
  hipLaunchKernelGGL(zero_word_kernel, dim3(1), dim3(1), 0, as_stream(stream), work);
  Q4_LAUNCHED("zero_word");
  const long grid = min((n + 4095) / 4096, 256L);
  hipLaunchKernelGGL(absmax_bits_kernel, dim3((unsigned)grid), dim3(1024), 0, as_stream(stream), sc32, n, work);
  Q4_LAUNCHED("absmax_bits");
  const long wgs = (long)(pad_rows(N) / PANEL) * ceil_div(nblk, 32);
  hipLaunchKernelGGL(e4m3_lift_kernel, dim3((unsigned)wgs), dim3(256), 0, as_stream(stream), sc32, N, nblk, work, sc8,
                     inv_dev);
  Q4_LAUNCHED("e4m3_lift");
  return Q4_OK;
}

int q4_w8_fold(const uint32_t* wq, const float* sc32, int N, int K, int8_t* W8, float* sw32, uint16_t* sw16,
               void* stream) {
  clear_error();
  if (int st = check_wk(N, K)) return st;
  Q4_ARG(wq && sc32 && W8, "null pointer");
  Q4_ARG(((uintptr_t)W8 & 15) == 0 && ((uintptr_t)wq & 15) == 0, "W8 and wq must be 16-byte aligned");
  const bool few = N < FOLD_ROWS;
  hipLaunchKernelGGL((few ? w8_fold_kernel<false, 2> : w8_fold_kernel<false, 8>), dim3(ceil_div(N, few ? 2 : 8)),
                     dim3(256), 0, as_stream(stream), reinterpret_cast<const uint4*>(wq), sc32, N, K, K / BLK, W8, sw32, sw16, 0);
  Q4_LAUNCHED("w8_fold");
  return Q4_OK;
}

int q4_w8_fold_packed(const uint32_t* wq, const float* sc32, int N, int K, int8_t* W8p, float* sw32, uint16_t* sw16,
                      void* stream) {
  clear_error();
  if (int st = check_wk(N, K)) return st;
  Q4_ARG(wq && sc32 && W8p, "null pointer");
  Q4_ARG(((uintptr_t)W8p & 15) == 0 && ((uintptr_t)wq & 15) == 0, "W8p and wq must be 16-byte aligned");
  const int rows = ceil_div(N, 32) * 32;
  const int kslices = (int)(q4_w8_packed_bytes(N, K) / ((size_t)rows * 32));
  const bool few = N < FOLD_ROWS;
  hipLaunchKernelGGL((few ? w8_fold_kernel<true, 2> : w8_fold_kernel<true, 8>), dim3(rows / (few ? 2 : 8)), dim3(256), 0,
                     as_stream(stream), reinterpret_cast<const uint4*>(wq), sc32, N, K, K / BLK, W8p, sw32, sw16, kslices);
  Q4_LAUNCHED("w8_fold_packed");
  return Q4_OK;
}

int q4_w4a8_ratio(const float* sc32, const float* sw32, int N, int K, uint16_t* ratio, void* stream) {
  clear_error();
  if (int st = check_wk(N, K)) return st;
  Q4_ARG(sc32 && sw32 && ratio, "null pointer");
  const int nblk = K / BLK;
  long units = (long)pad_rows(N) * nblk;
  hipLaunchKernelGGL(w4a8_ratio_kernel, dim3(ceil_div(units, 256)), dim3(256), 0, as_stream(stream), sc32, sw32, N,
                     nblk, ratio);
  Q4_LAUNCHED("w4a8_ratio");
  return Q4_OK;
}

int q4_repack_ref(const uint32_t* wp, const uint16_t* sc_ref, int N, int K, uint32_t* wq, uint16_t* sc_dev,
                  void* stream) {
  clear_error();
  if (int st = check_wk(N, K)) return st;
  Q4_ARG(N % 8 == 0, "reference layout needs N %% 8 == 0 (N=%d)", N);
  Q4_ARG((wp != nullptr) == (wq != nullptr), "wp and wq must both be given or both be NULL");
  Q4_ARG((sc_ref != nullptr) == (sc_dev != nullptr), "sc_ref and sc_dev must both be given or both be NULL");
  Q4_ARG(((uintptr_t)wq & 15) == 0, "wq must be 16-byte aligned");
  const int nblk = K / BLK;
  long units = (long)pad_rows(N) * nblk;
  hipLaunchKernelGGL(repack_ref_kernel, dim3(ceil_div(units, 256)), dim3(256), 0, as_stream(stream), wp, sc_ref, N, K,
                     nblk, reinterpret_cast<uint4*>(wq), sc_dev);
  Q4_LAUNCHED("repack_ref");
  return Q4_OK;
}

int q4_interleave_rows(const uint32_t* wa, const void* sa, const uint32_t* wb, const void* sb, int N, int K,
                       int scale_bytes, uint32_t* wout, void* sout, void* stream) {
  clear_error();
  if (int st = check_wk(N, K)) return st;
  Q4_ARG(wa && sa && wb && sb && wout && sout, "null pointer");
  Q4_ARG(N % 32 == 0, "interleaving needs N %% 32 == 0 (got N=%d)", N);
  Q4_ARG(scale_bytes == 1 || scale_bytes == 2, "scale_bytes must be 1 or 2");
  Q4_ARG(((uintptr_t)wa & 15) == 0 && ((uintptr_t)wb & 15) == 0 && ((uintptr_t)wout & 15) == 0,
         "weight words must be 16-byte aligned");
  const int nblk = K / BLK;
  const long units = (long)2 * N * nblk;
  hipLaunchKernelGGL(interleave_rows_kernel, dim3(ceil_div(units, 256)), dim3(256), 0, as_stream(stream),
                     reinterpret_cast<const uint4*>(wa), reinterpret_cast<const uint8_t*>(sa),
                     reinterpret_cast<const uint4*>(wb), reinterpret_cast<const uint8_t*>(sb), nblk, scale_bytes,
                     reinterpret_cast<uint4*>(wout), reinterpret_cast<uint8_t*>(sout), units);
  Q4_LAUNCHED("interleave_rows");
  return Q4_OK;
}

int q4_repack_e4m3_ref(const uint8_t* sc_ref, int N, int K, uint8_t* sc_dev, void* stream) {
  clear_error();
  if (int st = check_wk(N, K)) return st;
  Q4_ARG(sc_ref && sc_dev, "null pointer");
  const int nblk = K / BLK;
  long units = (long)pad_rows(N) * nblk;
  hipLaunchKernelGGL(repack_e4m3_ref_kernel, dim3(ceil_div(units, 256)), dim3(256), 0, as_stream(stream), sc_ref, N,
                     nblk, sc_dev);
  Q4_LAUNCHED("repack_e4m3_ref");
  return Q4_OK;
}

int q4_repack_w8_ref(const int8_t* w8_kn, int N, int K, int8_t* w8_nk, void* stream) {
  clear_error();
  Q4_ARG(N > 0 && K > 0, "bad shape N=%d K=%d", N, K);
  Q4_ARG(w8_kn && w8_nk, "null pointer");
  dim3 grid(ceil_div(N, 64), ceil_div(K, 64));
  hipLaunchKernelGGL(transpose_i8_kernel, grid, dim3(256), 0, as_stream(stream), w8_kn, K, N, w8_nk);
  Q4_LAUNCHED("repack_w8_ref");
  return Q4_OK;
}

}  // extern "C"
