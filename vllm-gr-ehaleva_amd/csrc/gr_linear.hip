// Projections of a decode step: out[t, n] = sum_k x[t, k] w[n, k] for up to a
// few hundred rows t (one per beam), bf16 / fp16 with float32 accumulation,
// optionally with the SwiGLU gate in the epilogue.
//
// What bounds it: at these row counts a projection has too few output tiles of
// the usual 256 x 256 for 256 CUs, and each CU is fed through 64 bytes per
// clock from its L2 and 128 from LDS.  So the tile is picked to give every CU
// one tile where that is possible (64 x 64 up to 128 x 192), and everything
// else hides latency:
//  * 64-deep stages of both operands go straight from global memory into LDS
//    (rows of 128 bytes, 16-byte chunks XOR-swizzled by the row), ST stages in
//    flight;
//  * 8 waves, 4 x 2 over the tile, two to a SIMD.  Every sum runs over k in
//    order through one accumulator, 32 at a time, as the library's kernels for
//    these shapes do: a split over depth inside the workgroup (less LDS traffic,
//    which does not bound it) measured the same and moved the decoder's logits
//    by as much as their own rounding error;
//  * the fragments of stage s + 1 are read while the MFMAs of stage s run; one
//    barrier per stage.
// What is left: 256 CUs read their tiles' operands, each for the first time in
// this launch, at 59 GB/s a CU; without the MFMAs the time is the same.  Deep
// projections on few columns (in 6144, out 2048) gain nothing over the library.
// Measured (bf16, weights cold, library -> this one, us; 2048 in):
//   rows              8            64           200          384          512
//   out 4096     11.6 ->  9.3  12.3 -> 12.0  13.8 -> 10.7  15.3 -> 16.0  17.8 -> 16.5
//   out 2048      8.2 ->  7.9   8.9 ->  8.5   9.6 ->  8.7  11.0 ->  9.1  11.4 ->  9.8
//   SwiGLU 6144  18.7 -> 13.2  20.4 -> 15.7  31.1 -> 22.9  37.8 -> 29.4  39.2 -> 32.8
//   out 8192     14.1 -> 11.5  14.8 -> 14.2  18.2 -> 16.0  24.4 -> 22.8  27.8 -> 24.1
// (SwiGLU against the library's product and the separate gate kernel.  The
// decoder leaves sizes like 384 rows x 4096 columns to the library.)
// All row tiles of a column tile run on one XCD: the weights, which come from
// HBM, are then read into one L2 only.
#include "gr_decoder.h"
#include "gr_mfma_tile.h"

#include <type_traits>

namespace gr {
namespace {

constexpr int LN_THREADS = 512;
constexpr int LN_BK = 64;  // depth of a stage: 128-byte rows

typedef float lf4_t __attribute__((__vector_size__(16)));

struct LinearArgs {
  void* out;
  int64_t out_stride;
  const void* x;
  int64_t x_stride;
  const void* w;
  int64_t w_stride;
  int M, N, K;  // N: output columns (the weights have 2 N rows with SWIGLU: gate, then up)
  int tiles_m, tiles_n;
  int out_f32;  // 0: the inputs' type; 1: float32; 2: float32 of the inputs' type
};

template <int DT> __device__ inline lf4_t mma32(u32x4_t a, u32x4_t b, lf4_t c) {
  if constexpr (DT == GR_DTYPE_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                  0, 0);
}

// This wave's LDS reads are done and all but its newest N transfers have
// landed (the compiler does not see the transfers), then the barrier.
template <int N> __device__ __forceinline__ void stage_barrier() {
  __asm__ volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int BM, int BN> constexpr int linear_stages() {
  return BM + BN <= 128 ? 8 : BM + BN <= 192 ? 6 : 4;
}

template <int DT, int BM, int BN, bool SWIGLU>
__global__ __launch_bounds__(LN_THREADS, 1) void linear_k(LinearArgs a) {
  constexpr int ST = linear_stages<BM, BN>();
  constexpr int STAGE = (BM + BN) * LN_BK * 2;  // bytes
  constexpr int LPS = (BM + BN) / 64;           // transfers per wave and stage (8 rows each)
  constexpr int FM = BM / 64, FN = BN / 32;     // 16-row fragments per wave of x and of w
  static_assert(!SWIGLU || FN % 2 == 0, "gate / up fragment pairs");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[ST * STAGE];
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int nt = (local / a.tiles_m) * 8 + xcd, mt = local % a.tiles_m;
  if (nt >= a.tiles_n) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = mt * BM, n0 = nt * (SWIGLU ? BN / 2 : BN);

  // transfer i of a stage moves LDS rows 8 (wave + 8 i) .. + 7 (x rows, then w
  // rows); lane l lands on row l >> 3, chunk l & 7 of them and fetches the
  // logical chunk (l & 7) ^ (row & 7).  Rows past the matrix repeat its last
  // (their results are not stored).  With SWIGLU, 16 gate rows and the 16 up
  // rows of the same columns alternate.
  const uint8_t* src[LPS];
#pragma unroll
  for (int i = 0; i < LPS; ++i) {
    const int row = 8 * (wave + 8 * i) + (lane >> 3);
    const int ch = (lane & 7) ^ (lane >> 3);
    const uint8_t* p;
    if (row < BM) {
      p = static_cast<const uint8_t*>(a.x) + (int64_t)min(m0 + row, a.M - 1) * a.x_stride * 2;
    } else {
      const int b = row - BM;
      const int n = SWIGLU ? min(n0 + (b >> 5) * 16 + (b & 15), a.N - 1) + ((b >> 4) & 1) * a.N : min(n0 + b, a.N - 1);
      p = static_cast<const uint8_t*>(a.w) + (int64_t)n * a.w_stride * 2;
    }
    src[i] = p + ch * 16;
  }
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(lds);
  auto fetch = [&](int s, int buf) {
#pragma unroll
    for (int i = 0; i < LPS; ++i)
      dma_v(lds0 + (uint32_t)(buf * STAGE + (wave + 8 * i) * 1024), src[i] + (int64_t)s * (LN_BK * 2));
  };
  struct Frags { u32x4_t x[2][FM], w[2][FN]; };  // the stage's two 32-deep steps
  // chunk 4 h + lane / 16 of the fragments' row lane % 16, h = step
  const int r16 = lane & 15;
  const int fch0 = ((lane >> 4) ^ (r16 & 7)) * 16, fch1 = ((4 + (lane >> 4)) ^ (r16 & 7)) * 16;
  const int xo = (wm * (BM / 4) + r16) * 128, wo = (BM + wn * (BN / 2) + r16) * 128;
  auto read = [&](int buf, Frags& f) __attribute__((always_inline)) {
    const uint8_t* p = lds + buf * STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int fch = h ? fch1 : fch0;
#pragma unroll
      for (int j = 0; j < FM; ++j) f.x[h][j] = *reinterpret_cast<const u32x4_t*>(p + xo + fch + j * 2048);
#pragma unroll
      for (int i = 0; i < FN; ++i) f.w[h][i] = *reinterpret_cast<const u32x4_t*>(p + wo + fch + i * 2048);
    }
  };
  lf4_t acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = lf4_t{0.f, 0.f, 0.f, 0.f};
  auto mul = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = mma32<DT>(f.w[h][i], f.x[h][j], acc[i][j]);
  };

  const int n = a.K / LN_BK;  // >= ST
#pragma unroll
  for (int s = 0; s < ST; ++s) fetch(s, s);
  stage_barrier<(ST - 1) * LPS>();
  Frags fa, fb;
  read(0, fa);
  // stage s: its fragments are in registers (its buffer, s % ST, is free once
  // every wave is past the barrier); stage s + 1 has landed at the barrier,
  // stages s + 2 .. s + ST - 1 may be in flight
  int buf = 0;
  auto step = [&](int s, const Frags& cur, Frags& nxt) __attribute__((always_inline)) {
    stage_barrier<(ST - 2) * LPS>();
    const int nb = buf + 1 == ST ? 0 : buf + 1;
    read(nb, nxt);
    fetch(s + ST, buf);
    buf = nb;
    __builtin_amdgcn_sched_barrier(0);  // the reads go out ahead of the MFMAs
    mul(cur);
  };
  int s = 0;
  for (; s + 1 < n - ST; s += 2) {
    step(s, fa, fb);
    step(s + 1, fb, fa);
  }
  if (s < n - ST) {
    step(s, fa, fb);
    fa = fb;
  }
  // the last ST stages: nothing more to fetch, one stage fewer in flight each time
  auto tail = [&](auto left, const Frags& cur, Frags& nxt) __attribute__((always_inline)) {
    constexpr int L = decltype(left)::value;  // stages after this one
    if constexpr (L > 0) {
      stage_barrier<(L - 1) * LPS>();
      const int nb = buf + 1 == ST ? 0 : buf + 1;
      read(nb, nxt);
      buf = nb;
      __builtin_amdgcn_sched_barrier(0);
    }
    mul(cur);
  };
#define LN_TAIL(L) \
  if constexpr (ST > L) tail(std::integral_constant<int, L>{}, (ST - 1 - L) % 2 ? fb : fa, (ST - 1 - L) % 2 ? fa : fb);
  LN_TAIL(7) LN_TAIL(6) LN_TAIL(5) LN_TAIL(4) LN_TAIL(3) LN_TAIL(2) LN_TAIL(1) LN_TAIL(0)
#undef LN_TAIL

  using S = uint16_t;
  // fragment (i, j), register u: column 16 i + 4 (lane / 16) + u, row 16 j + lane % 16
  auto put = [&](int t, int col, const float (&v)[4]) {
    if (t >= a.M || col >= a.N) return;
    if (a.out_f32) {
      lf4_t f = {v[0], v[1], v[2], v[3]};
      if (a.out_f32 == 2) {
#pragma unroll
        for (int u = 0; u < 4; ++u) f[u] = Elem<DT>::to_float(Elem<DT>::from_float(f[u]));
      }
      *reinterpret_cast<lf4_t*>(static_cast<float*>(a.out) + (int64_t)t * a.out_stride + col) = f;
    } else {
      *reinterpret_cast<u32x2_t*>(static_cast<S*>(a.out) + (int64_t)t * a.out_stride + col) =
          u32x2_t{Mma<DT>::pack2(v[0], v[1]), Mma<DT>::pack2(v[2], v[3])};
    }
  };
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    const int t = m0 + wm * (BM / 4) + j * 16 + r16;
    if constexpr (SWIGLU) {
#pragma unroll
      for (int i = 0; i < FN; i += 2) {
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          // (rounded as the gate kernel reads them: a decode step's results then
          // differ from the two-kernel form's by summation order only)
          const float g = Elem<DT>::to_float(Elem<DT>::from_float(acc[i][j][u]));
          const float up = Elem<DT>::to_float(Elem<DT>::from_float(acc[i + 1][j][u]));
          v[u] = g / (1.0f + __expf(-g)) * up;
        }
        put(t, n0 + wn * (BN / 4) + i * 8 + 4 * (lane >> 4), v);
      }
    } else {
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        put(t, n0 + wn * (BN / 2) + i * 16 + 4 * (lane >> 4), v);
      }
    }
  }
}

// The tile with the least estimated time: rounds of workgroups on the XCD that
// gets the most of them (one to a CU, 32 CUs; column tiles go round the XCDs
// whole), each a fixed part and its stages.  Nanoseconds of both by least
// squares over 550 to 940 one-round launches a tile (64 tiles and more; 1 to 512
// rows, 512 to 16384 weight rows, 8 to 32 stages; rms residual 1.1 to 2.3 us).
// The fixed part holds the launch, the first stages' way into LDS and the
// stores; a stage is 25 to 27 bytes per clock into the CU.  On 1428 other random
// sizes the pick is within 3 % of the fastest of the four tiles.  Rounds over
// the whole chip's 256 CUs instead take 7 x 34 tiles (448 rows, 2160 columns)
// for one round, though two XCDs get 35 of them: 13.3 us against 10.3.
struct LinearTile { int bm, bn, fixed, stage; };
constexpr LinearTile kLinearTiles[] = {
    {64, 64, 2900, 260}, {128, 64, 3300, 350}, {128, 128, 4200, 520}, {128, 192, 5300, 680}};

int pick_linear_tile(int M, int rows_w, int K) {
  int best = 0;
  int64_t cost = INT64_MAX;
  for (int i = 0; i < 4; ++i) {
    const LinearTile& t = kLinearTiles[i];
    const int64_t per_xcd = (int64_t)((M + t.bm - 1) / t.bm) * (((rows_w + t.bn - 1) / t.bn + 7) / 8);
    const int64_t c = (per_xcd + 31) / 32 * (t.fixed + (int64_t)(K / LN_BK) * t.stage);
    if (c < cost) {
      cost = c;
      best = i;
    }
  }
  return best;
}

template <int DT, int BM, int BN, bool SWIGLU>
void launch_linear(LinearArgs a, hipStream_t stream) {
  a.tiles_m = (a.M + BM - 1) / BM;
  const int bn = SWIGLU ? BN / 2 : BN;
  a.tiles_n = (a.N + bn - 1) / bn;
  const dim3 grid((unsigned)((a.tiles_n + 7) / 8 * 8 * a.tiles_m));
  hipLaunchKernelGGL((linear_k<DT, BM, BN, SWIGLU>), grid, dim3(LN_THREADS), 0, stream, a);
}

template <int DT, bool SWIGLU>
void launch_linear_tile(const LinearArgs& a, hipStream_t stream) {
  switch (pick_linear_tile(a.M, SWIGLU ? 2 * a.N : a.N, a.K)) {
    case 0: launch_linear<DT, 64, 64, SWIGLU>(a, stream); break;
    case 1: launch_linear<DT, 128, 64, SWIGLU>(a, stream); break;
    case 2: launch_linear<DT, 128, 128, SWIGLU>(a, stream); break;
    default: launch_linear<DT, 128, 192, SWIGLU>(a, stream); break;
  }
}

}  // namespace
}  // namespace gr

using namespace gr;

extern "C" int gr_linear_tile(int num_tokens, int out_features, int in_features, int swiglu) {
  if (num_tokens < 1 || out_features < 1 || out_features > (1 << 28) || in_features < 1) return 0;
  const LinearTile& t = kLinearTiles[pick_linear_tile(num_tokens, (swiglu ? 2 : 1) * out_features, in_features)];
  return t.bm * 1000 + t.bn;
}

extern "C" gr_status_t gr_linear(void* out, int64_t out_stride, const void* x, int64_t x_stride, const void* w,
                                 int64_t w_stride, int num_tokens, int out_features, int in_features, int swiglu,
                                 int out_f32, int dtype, hipStream_t stream) {
  if (num_tokens < 0 || out_features < 1 || in_features < 1 || (swiglu != 0 && swiglu != 1) ||
      out_f32 < 0 || out_f32 > 2 || !dtype_valid(dtype))
    return GR_ERR_INVALID_ARG;
  if (num_tokens == 0) return GR_OK;
  if (!out || !x || !w || out_stride < out_features || x_stride < in_features || w_stride < in_features)
    return GR_ERR_INVALID_ARG;
  auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  // whole 16-byte chunks of every row, whole fragments of columns, at least
  // as many stages as the deepest pipeline holds
  if (dtype == GR_DTYPE_F32 || in_features % LN_BK != 0 || in_features < 8 * LN_BK || out_features % 16 != 0 ||
      out_features > (1 << 28) || !al(x) || !al(w) || !al(out) || x_stride % 8 != 0 || w_stride % 8 != 0 ||
      out_stride % 4 != 0 || num_tokens > 65536)
    return GR_ERR_UNSUPPORTED;
  LinearArgs a{out, out_stride, x, x_stride, w, w_stride, num_tokens, out_features, in_features, 0, 0, out_f32};
  if (dtype == GR_DTYPE_BF16) {
    if (swiglu) launch_linear_tile<GR_DTYPE_BF16, true>(a, stream);
    else launch_linear_tile<GR_DTYPE_BF16, false>(a, stream);
  } else {
    if (swiglu) launch_linear_tile<GR_DTYPE_F16, true>(a, stream);
    else launch_linear_tile<GR_DTYPE_F16, false>(a, stream);
  }
  return launch_status();
}
