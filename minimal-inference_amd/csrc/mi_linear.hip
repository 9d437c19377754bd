// Linear layers of few rows (decode steps): out = x W^T (+ bias), bf16 with
// fp32 accumulation and one rounding.
//
// Reference: the projections of Attention.forward (model.py:160-163, 245-252),
// the MLP (model.py:301-311) and the LM head (model.py:432-435), which decode
// steps call with one row per request.
//
// Bound: HBM, the one read of W.  A workgroup of 4 waves owns 16 R rows of W
// (output columns) over all of K, so nothing is exchanged between workgroups
// and no workspace is needed.  The waves split K: at each step wave w takes
// one slab of 64 k (128 bytes of each row) of the W rows and of x.  Its loads
// cover whole 128-byte lines of 8 rows each (the MFMA operand layout would
// touch 16 lines per quarter wave, four times over), D steps ahead in
// registers -- LDS could hold two or three steps -- and pass through a
// wave-private LDS slot into operand order, so the waves meet only once, at the
// end, where their accumulators are added in wave order through LDS: the
// result does not depend on timing.  Per slab, 16 rows of W and 16 of x: two
// 16x16x32 MFMAs with W as A and x^T as B.
#include "mi_common.h"

namespace {

constexpr int kWaves = 4;
constexpr int kSlab = 64;             // k per slab
constexpr int kSlabBytes = kSlab * 2;  // of one row
constexpr int kMaxRows = 32;
constexpr int kMaxK = 1 << 23;  // the byte size of a workgroup's rows of W (up to 64) is an int
constexpr int kBufferWord3 = 0x00020000;
// Cache-policy operand of the buffer intrinsics: nt (non-temporal / streaming).
constexpr int kCacheNT = 2;

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2_t;
typedef __attribute__((address_space(3))) char lds_t;

struct LinearParams {
  const uint16_t* x;
  int64_t x_stride;
  const uint16_t* w;
  const uint16_t* bias;  // null: none
  uint16_t* out;
  int64_t o_stride;
  int rows, n, k;  // n: columns of out
};

__device__ __forceinline__ u32x4_t lds_load16(const lds_t* p) {
  return *(const __attribute__((address_space(3))) u32x4_t*)p;
}
__device__ __forceinline__ void lds_store16(lds_t* p, u32x4_t v) { *(__attribute__((address_space(3))) u32x4_t*)p = v; }
// Slot of 16-byte chunk c in a staged row: two 128-byte rows make one period
// of the LDS banks, so the 16 rows an MFMA operand read touches at one chunk
// fall on distinct banks.
__device__ __forceinline__ int chunk_slot(int r, int c) { return c ^ ((r >> 1) & 7); }

template <int R, int MB, int D>
struct LinearTraits {
  static constexpr int SLOT = (R + MB) * 16 * kSlabBytes;  // one wave's slab of W and x
  static constexpr int RED = R * MB * 1024;                // its accumulators
  static constexpr int SMEM = kWaves * (SLOT > RED ? SLOT : RED);
  static_assert(SMEM <= 160 * 1024, "LDS");
};

// GLU: W holds n gate rows, then n up rows; tile r is the gate's (even r) or the
// up part's (odd) of the output columns 16 (r / 2) .., and out = silu(gate) * up,
// rounded where the separate kernel rounds.  It saves that launch (of eight rows'
// 3.5 us) and the write and read of gate and up.
//
// HALF: only the first 8 rows of the one tile, for weights of so few rows that
// most CUs had no workgroup.  The matrix instructions' other 8 rows hold what is
// in LDS and are not written out.
template <int R, int MB, int D, bool GLU, bool HALF>
__global__ __launch_bounds__(64 * kWaves) void linear_kernel(LinearParams p) {
  constexpr int HALVES = GLU ? 2 : 1, COLS = HALF ? 8 : 16 * R / HALVES;  // output columns of a workgroup
  static_assert(R % HALVES == 0, "gate and up tiles in pairs");
  static_assert(!HALF || (R == 1 && !GLU), "half of one tile");
  constexpr int WL = HALF ? 1 : 2 * R;  // loads of 8 rows of W per slab
  using T = LinearTraits<R, MB, D>;
  __shared__ __attribute__((aligned(16))) char smem[T::SMEM];
  lds_t* const lds = (lds_t*)smem;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const int row0 = int(blockIdx.x) * COLS;
  const int nslab = p.k / kSlab, steps = (nslab - w + kWaves - 1) / kWaves;  // this wave's: w, w + 4, ...

  // load i of a slab: 8 rows, lane l chunk l % 8 of row l / 8; rows past the
  // end read out of range: zeros
  const char* wbase = reinterpret_cast<const char*>(p.w) + int64_t(row0) * p.k * 2;
  const int wsize = min(COLS, p.n - row0) * p.k * 2;  // of each half
  const int64_t up = int64_t(p.n) * p.k * 2;
  const int xsize = int(((p.rows - 1) * p.x_stride + p.k) * 2);
  const int lr = lane / 8, lc = (lane % 8) * 16;
  const int wv = lr * p.k * 2 + lc, wrow8 = 8 * p.k * 2;
  const int xv = int(lr * p.x_stride * 2) + lc, xrow8 = int(8 * p.x_stride * 2);
  u32x4_t wr[D][WL], xr[D][2 * MB];
  auto load = [&](int d, int step) {
    const int off = (step * kWaves + w) * kSlabBytes;
    const bool ok = step < steps;
    __amdgpu_buffer_rsrc_t rw[HALVES];
#pragma unroll
    for (int h = 0; h < HALVES; ++h)
      rw[h] = __builtin_amdgcn_make_buffer_rsrc((void*)(wbase + h * up + off), (short)0, ok ? wsize - off : 0,
                                                kBufferWord3);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(reinterpret_cast<const char*>(p.x) + off), (short)0, ok ? xsize - off : 0, kBufferWord3);
    // W is read once: non-temporal
#pragma unroll
    for (int i = 0; i < WL; ++i)
      wr[d][i] = __builtin_amdgcn_raw_buffer_load_b128(
          rw[(i / 2) % HALVES], wv + (i / 2 / HALVES * 2 + i % 2) * wrow8, 0, kCacheNT);
#pragma unroll
    for (int i = 0; i < 2 * MB; ++i) xr[d][i] = __builtin_amdgcn_raw_buffer_load_b128(rx, xv + i * xrow8, 0, 0);
  };

  mi::f32x4_t acc[R][MB];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[r][b] = mi::f32x4_t{0.f, 0.f, 0.f, 0.f};
  lds_t* const slot = lds + w * T::SLOT;
  // staged row 8 i + lr: its permutation depends on the row modulo 16
  int so[2], ro[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) so[i] = lr * kSlabBytes + chunk_slot(8 * i + lr, lane % 8) * 16;
#pragma unroll
  for (int s = 0; s < 2; ++s) ro[s] = n * kSlabBytes + chunk_slot(n, 4 * s + g) * 16;  // operand chunk 4 s + g of row n

  // issued in the order they are waited for, here and in the loop
#pragma unroll
  for (int d = 0; d < D; ++d) {
    load(d, d);
    __builtin_amdgcn_sched_barrier(0);
  }
  // (no branch inside a round of D steps, so that the compiler's wait before a
  // step is exactly "the D - 1 later ones in flight"; the steps past the last
  // one add zeros)
  for (int s0 = 0; s0 < steps; s0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
      for (int i = 0; i < WL; ++i) lds_store16(slot + i * 1024 + so[i & 1], wr[d][i]);
#pragma unroll
      for (int i = 0; i < 2 * MB; ++i) lds_store16(slot + (2 * R + i) * 1024 + so[i & 1], xr[d][i]);
      load(d, s0 + d + D);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        mi::bf16x8_t a[R], x[MB];
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = __builtin_bit_cast(mi::bf16x8_t, lds_load16(slot + r * 2048 + ro[s]));
#pragma unroll
        for (int b = 0; b < MB; ++b)
          x[b] = __builtin_bit_cast(mi::bf16x8_t, lds_load16(slot + (R + b) * 2048 + ro[s]));
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int b = 0; b < MB; ++b) acc[r][b] = mi::mfma_16x16x32_bf16(a[r], x[b], acc[r][b]);
      }
      // (left alone, the scheduler gathers the LDS stores of the whole round
      // at its start and waits for every load there)
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // the waves' accumulators through LDS; wave w adds the blocks w, w + 4, ...
  // Lane (g, n) holds columns 4 g .. 4 g + 3 of the output of row 16 b + n.
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int b = 0; b < MB; ++b)
      lds_store16(lds + (w * R * MB + r * MB + b) * 1024 + lane * 16, __builtin_bit_cast(u32x4_t, acc[r][b]));
  __syncthreads();
  auto total = [&](int q) {
    mi::f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int o = 0; o < kWaves; ++o)
      sum += __builtin_bit_cast(mi::f32x4_t, lds_load16(lds + (o * R * MB + q) * 1024 + lane * 16));
    return sum;
  };
  for (int q = w; q < R / HALVES * MB; q += kWaves) {
    const int r = q / MB, b = q - r * MB;  // r: the tile (or pair of tiles)
    mi::f32x4_t sum = total(HALVES * r * MB + b);
    const int m = b * 16 + n, col = row0 + r * 16 + 4 * g;
    if (m < p.rows && row0 + r * 16 < p.n && (!HALF || g < 2)) {
      if (p.bias) {
        const u32x2_t bb = *reinterpret_cast<const u32x2_t*>(p.bias + col);
        sum[0] += mi::bf16_lo(bb.x);
        sum[1] += mi::bf16_hi(bb.x);
        sum[2] += mi::bf16_lo(bb.y);
        sum[3] += mi::bf16_hi(bb.y);
      }
      u32x2_t v = {mi::cvt_pk_bf16(sum[0], sum[1]), mi::cvt_pk_bf16(sum[2], sum[3])};
      if constexpr (GLU) {
        const mi::f32x4_t u = total((HALVES * r + 1) * MB + b);
        v[0] = mi::silu_mul_bf16x2(v[0], mi::cvt_pk_bf16(u[0], u[1]));
        v[1] = mi::silu_mul_bf16x2(v[1], mi::cvt_pk_bf16(u[2], u[3]));
      }
      *reinterpret_cast<u32x2_t*>(p.out + int64_t(m) * p.o_stride + col) = v;
    }
  }
}

typedef void (*LinearKernel)(LinearParams);

// The form of a launch, from the 16-row tiles of W and the 16-row blocks of x
// (us at 8 / 32 rows, weights rotated through 600 MB; library = the hipBLASLt
// kernel torch picks):
//                        R 1 D 4      R 1 D 2      R 2 D 2      R 4 D 2    library
//   N   896 K   896     3.2 /  4.2   3.3 /  4.0   3.8 /  4.7   4.9 /  6.3   5.5 / 7.5
//   N   896 K  4864     6.8 / 10.7   8.0 / 10.3   9.8 / 13.7  15.7 / 19.9    17 / 13
//   N  4096 K  4096     8.2 / 10.4   8.7 / 10.0  10.6 / 12.8  14.1 / 17.4    16 / 13
//   N  4096 K 14336    23.1 / 35.0  26.4 / 34.1  33.0 / 41.6  46.0 / 56.7    26 / 31
//   N  6144 K  4096    12.9 / 17.4  12.0 / 16.8  13.0 / 14.2  17.0 / 18.4    14 / 15
//   N 28672 K  4096    41.2 / 61.6  40.3 / 60.2  48.1 / 53.6  43.5 / 46.4    62 / 55
//   N 151936 K  896    60.4 / 87.2  51.2 / 78.0  43.6 / 63.4  44.9 / 55.0    53 / 65
// One tile per workgroup while x is one block: its re-reads by every workgroup
// are then no more than W.  With up to one tile per CU the loads in flight of a
// workgroup bound it (D 4, as for long K); two tiles when the launch is so long
// that starting and ending workgroups shows.  With two blocks of x, what bounds
// it is x from L2, so as many tiles as still leave workgroups for the CUs (512 tiles
// in fours leave half of them idle: 8,192 x 7,168, 32 rows, 29.5 us, library 25.7).
// Half tiles up to 128 tiles (full ones leave half of the CUs or more idle), with
// two blocks of x, which they read twice as often, for long k only (us at 8 / 32 rows,
// whole / half): 896 x 4,864 6.8 / 10.3, 5.6 / 9.2; 2,048 x 8,960 11.4 / 18.1, 9.1 / 15.7;
// 1,024 x 3,072 5.1 / 7.4, 4.3 / 6.7; 1,536 x 1,536 4.1 / 5.0, 3.8 / 5.3; 896 x 896
// 3.2 / 4.0, 3.05 / 4.0.  (8 waves, or D 8, with either: slower.)
template <int R, int D, bool GLU = false, bool HALF = false>
LinearKernel pick(int mb) { return mb == 1 ? linear_kernel<R, 1, D, GLU, HALF> : linear_kernel<R, 2, D, GLU, HALF>; }

LinearKernel pick_kernel(int tiles, int k, int mb, int* cols) {
  if (tiles <= 128 && (mb == 1 || k >= 2048)) {
    *cols = 8;
    return pick<1, 4, false, true>(mb);
  }
  const int r = mb == 1 ? (tiles > 2048 ? 2 : 1) : tiles <= 256 ? 1 : tiles <= 512 ? 2 : 4;
  *cols = 16 * r;
  if (mb == 1 && (r == 2 || (tiles > 256 && k < 8192))) return r == 2 ? pick<2, 2>(1) : pick<1, 2>(1);
  if (mb == 1) return linear_kernel<1, 1, 4, false, false>;
  return r == 1 ? pick<1, 2>(2) : r == 2 ? pick<2, 2>(2) : linear_kernel<4, 2, 2, false, false>;
}

// With the gated product, from the pairs of a gate and an up tile (us at 8 / 32
// rows; separate = the forms above and the SiLU kernel after them):
//                      pairs       R 2          R 4       separate
//   N  9728 K   896      304    6.6 /  8.1   5.9 /  6.9   8.6 /  9.2
//   N  9728 K  4096      304   19.4 / 23.3  19.4 / 20.2  20.4 / 22.3
//   N 19456 K  2048      608   16.5 / 20.1  20.2 / 22.5  20.4 / 24.9
//   N 28672 K  4096      896   39.2 / 47.8  42.6 / 43.6  41.1 / 46.8
//   N 37888 K  3584     1184   43.5 / 53.9  46.9 / 52.0  44.9 / 55.5
// Two pairs where that costs no CU more tiles (fewer reads of x): of a launch of
// one round, and with two blocks of x of any.  (D 4 is slower on all but 59,136 x
// 8,192, where it is equal.)
LinearKernel pick_glu(int pairs, int mb, int* cols) {
  const bool even = ((pairs + 1) / 2 + 255) / 256 * 2 <= (pairs + 255) / 256;
  const bool two = even && (mb == 2 || pairs <= 512);
  *cols = two ? 32 : 16;
  return two ? pick<4, 2, true>(mb) : pick<2, 2, true>(mb);
}

// Both entry points; `halves` 2: gate and up rows, n output columns.
int launch_linear(const char* name, const void* x, int64_t x_stride, const void* weight, const void* bias, void* out,
                  int64_t out_stride, int32_t rows, int32_t n, int32_t k, int halves, mi_stream_t stream) {
  mi::clear_error();
  if (rows < 0 || rows > kMaxRows || n <= 0 || n % 16 || k <= 0 || k % kSlab || k > kMaxK)
    return mi::fail(MI_ERR_INVALID, "%s: rows %d (0..%d), n %d (multiple of 16), k %d (multiple of %d, at most %d)", name,
                    rows, kMaxRows, n, k, kSlab, kMaxK);
  if (rows == 0) return MI_OK;
  if (!x || !weight || !out) return mi::fail(MI_ERR_INVALID, "%s: null pointer argument", name);
  if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(weight) & 15) ||
      (reinterpret_cast<uintptr_t>(bias) & 7) || (reinterpret_cast<uintptr_t>(out) & 7) || x_stride % 8 || out_stride % 4)
    return mi::fail(MI_ERR_INVALID, "%s: x rows and weight must be 16-byte, bias and out rows 8-byte aligned", name);
  if (x_stride < k || out_stride < n || int64_t(rows) * x_stride > (1 << 29))
    return mi::fail(MI_ERR_INVALID, "%s: row strides %lld / %lld for k %d, n %d", name, (long long)x_stride,
                    (long long)out_stride, k, n);
  LinearParams p;
  p.x = static_cast<const uint16_t*>(x);
  p.x_stride = x_stride;
  p.w = static_cast<const uint16_t*>(weight);
  p.bias = static_cast<const uint16_t*>(bias);
  p.out = static_cast<uint16_t*>(out);
  p.o_stride = out_stride;
  p.rows = rows;
  p.n = n;
  p.k = k;
  const int mb = (rows + 15) / 16;
  int cols = 16;  // output columns of a workgroup
  const LinearKernel kernel = halves == 2 ? pick_glu(n / 16, mb, &cols) : pick_kernel(n / 16, k, mb, &cols);
  hipLaunchKernelGGL(kernel, dim3((n + cols - 1) / cols), dim3(64 * kWaves), 0, static_cast<hipStream_t>(stream), p);
  return mi::check_launch("linear_kernel");
}

}  // namespace

extern "C" int mi_linear(const void* x, int64_t x_stride, const void* weight, const void* bias, void* out,
                         int64_t out_stride, int32_t rows, int32_t n, int32_t k, mi_stream_t stream) {
  return launch_linear("linear", x, x_stride, weight, bias, out, out_stride, rows, n, k, 1, stream);
}

extern "C" int mi_linear_silu(const void* x, int64_t x_stride, const void* weight, void* out, int64_t out_stride,
                              int32_t rows, int32_t n, int32_t k, mi_stream_t stream) {
  return launch_linear("linear_silu", x, x_stride, weight, nullptr, out, out_stride, rows, n, k, 2, stream);
}
