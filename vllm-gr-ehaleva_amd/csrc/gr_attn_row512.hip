// BeamAttention decode on the matrix cores for 512-byte K / V rows (float32 at
// head_dim 128, bf16 / fp16 at head_dim 256), in float32 precision throughout.
//
// What bounds it: these shapes are small (tens of megabytes of KV at most a
// request), so the time is the chain of one workgroup: per tile of a wave the
// loads of V, then of the next K (each CU takes its 1.1 MB at 45 GB/s in the
// head_dim 256 case below; streams reach 95 and more), or, in float32, the
// float32 MFMA rate.
// The split is therefore over rows and, inside the workgroup, over keys: a
// workgroup owns 16 query rows of one (request, KV head) -- the smallest MFMA
// tile, for the most workgroups -- and its 8 waves take every eighth tile of 32
// keys, each with its own online softmax; the eight partial states meet in LDS
// at the end.  No second launch and no workspace.  Workgroups of one (request,
// KV head) sit on one XCD and share its L2.
//
// Formulation (v_mfma_f32_16x16x32_{bf16,f16}, v_mfma_f32_16x16x4_f32), lane =
// (quarter g, m = lane % 16):
//   S^T[key][row] = K . Q^T   A = K rows from LDS, B = Q rows (registers)
//   O^T[d][row]  += V^T . P^T A = V (registers), B = P as the S^T accumulators hold it
// The contraction index of an MFMA may be numbered at will as long as both
// operands agree, which saves every layout change but one:
//  * QK: step j contracts the 16-byte chunks 4 j + g of a row;
//  * PV: an accumulator register (block kb, r) of quarter g is key 16 kb + 4 g +
//    r, so a lane loads V rows of exactly these keys (8 of the tile's 32), 16
//    bytes at chunk 16 c + m, and output block (c, e) is dim PER (16 c + m) + e.
//    float32 values are operands as loaded; 16-bit ones need an 8 x 8 transpose
//    inside the lane (32 byte permutes per chunk).
// K tiles go straight from global memory into the wave's own LDS tile (chunks
// XOR-swizzled by the key, so the A reads touch every bank once; the 16-bit
// merge's writes at the end take 4 cycles more each than they need); the next
// tile's transfer runs under this tile's softmax and PV, and V arrives in
// registers under QK.  No barrier inside the loop: a wave reads only its own
// tiles.
//
// Measured (MI355X, whole call, the generic kernel -> this one): float32, 1
// request x 32 beams, 512-token prompt, 16 / 4 heads: 174 -> 21.4 us; bf16
// head_dim 256, 4 requests x 64 beams, 1024-token prompts, 16 / 8 heads, soft
// cap: 557 -> 26.2 us (24.7 with two terms a weight); fp16, the same without the
// cap: 551 -> 28.6 us (43.4 where every tile takes the float32 MFMA).  Error
// against float64: 5.7e-7 -> 4.2e-7 and 1.7e-3 (output rounding) both.
//
// Precision: scores, probabilities and sums are float32, and PV takes all 24
// bits of a probability: as three 16-bit terms (three MFMAs), and in fp16, whose
// range they would leave, a tile with a probability below 2^-12 of the largest
// through the float32 MFMA.
#include "gr_mfma_tile.h"

namespace gr {
namespace {

constexpr int R5_THREADS = 512;
constexpr int R5_WAVES = R5_THREADS / 64;
constexpr int R5_ROWS = 16;      // query rows per workgroup
constexpr int R5_KEYS = 32;      // keys per wave tile
constexpr int R5_BYTES = 512;    // one K / V row
constexpr int R5_TILE = R5_KEYS * R5_BYTES;

typedef float f4_t __attribute__((__vector_size__(16)));

template <int DT> struct Row512;
template <> struct Row512<GR_DTYPE_F32> {
  static constexpr int PER = 4;  // elements per 16-byte chunk
  static constexpr float PSCALE = 1.f;  // PV takes its weights times this
  __device__ static inline f4_t qk(u32x4_t k, u32x4_t q, f4_t s) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(k[e]), __uint_as_float(q[e]), s, 0, 0, 0);
    return s;
  }
  // element e of a V chunk
  __device__ static inline float v_elem(u32x4_t v, int e) { return __uint_as_float(v[e]); }
  __device__ static inline u32x4_t pack(const float (&v)[4]) {
    return u32x4_t{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
  }
};
template <> struct Row512<GR_DTYPE_BF16> {
  static constexpr int PER = 8;
  static constexpr float PSCALE = 1.f;
  static constexpr uint32_t HEAD = 0xffff0000u;  // sign, exponent and the leading 8 bits of a float32
  static constexpr float TERM_MIN = 0x1p-126f;   // the smallest normal value of a term
  __device__ static inline f4_t mma(u32x4_t a, u32x4_t b, f4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  }
  __device__ static inline f4_t qk(u32x4_t k, u32x4_t q, f4_t s) { return mma(k, q, s); }
  __device__ static inline u32x4_t pack(const float (&v)[8]) {
    return u32x4_t{Mma<GR_DTYPE_BF16>::pack2(v[0], v[1]), Mma<GR_DTYPE_BF16>::pack2(v[2], v[3]),
                   Mma<GR_DTYPE_BF16>::pack2(v[4], v[5]), Mma<GR_DTYPE_BF16>::pack2(v[6], v[7])};
  }
};
template <> struct Row512<GR_DTYPE_F16> {
  static constexpr int PER = 8;
  static constexpr float PSCALE = 0x1p15f;       // the largest weight near the top of fp16's range
  static constexpr uint32_t HEAD = 0xffffe000u;  // ... and the leading 11 bits
  static constexpr float TERM_MIN = 0x1p-24f;    // fp16's smallest value
  // Scaled weights from 8 are sums of three terms: their last bit is 2^-20 or
  // more, and a term raised to TERM_MIN adds 2^-27 of them at most.
  static constexpr float SPLIT_MIN = 8.f;
  __device__ static inline f4_t mma(u32x4_t a, u32x4_t b, f4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                  0, 0);
  }
  __device__ static inline f4_t qk(u32x4_t k, u32x4_t q, f4_t s) { return mma(k, q, s); }
  __device__ static inline float v_elem(u32x4_t v, int e) {
    return Elem<GR_DTYPE_F16>::to_float((uint16_t)(v[e >> 1] >> (16 * (e & 1))));
  }
  __device__ static inline u32x4_t pack(const float (&v)[8]) {
    return u32x4_t{Mma<GR_DTYPE_F16>::pack2(v[0], v[1]), Mma<GR_DTYPE_F16>::pack2(v[2], v[3]),
                   Mma<GR_DTYPE_F16>::pack2(v[4], v[5]), Mma<GR_DTYPE_F16>::pack2(v[6], v[7])};
  }
};

// A weight as three terms of the type, each the leading bits of what is left:
// all 24 bits of it.  A term that would be zero beside p > 0 is raised to
// TERM_MIN, so that an infinite V row gives the infinity that a float32 weight
// gives it, not 0 * infinity.
template <int DT> __device__ inline void split_weight(float p, float (&t)[3]) {
  using M = Row512<DT>;
  const float lo = p > 0.f ? M::TERM_MIN : 0.f;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float h = __uint_as_float(__float_as_uint(p) & M::HEAD);
    t[i] = fmaxf(h, lo);
    p -= h;
  }
}

// The row's partial outputs of one wave in LDS: 16 rows of PER * 32 floats, 16
// bytes of padding a row (rows start on different banks).
template <int PER> constexpr int r5_pitch() { return PER * 32 + 4; }
template <int PER> constexpr int r5_region() {
  return R5_ROWS * r5_pitch<PER>() * 4 > R5_TILE ? R5_ROWS * r5_pitch<PER>() * 4 : R5_TILE;
}

// A wait that no memory access crosses, in the compiler or the schedule:
// gfx9 s_waitcnt immediates (vmcnt in bits 3:0 and 15:14, lgkmcnt in 11:8).
constexpr int WAIT_VM16 = 0x4F70;  // at most 16 vector-memory operations outstanding
constexpr int WAIT_ALL = 0x0070;   // none, and no LDS or scalar read
template <int IMM> __device__ __forceinline__ void fence() {
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(IMM);
  __builtin_amdgcn_sched_barrier(0);
  __asm__ volatile("" ::: "memory");
}

// Same rows, keys, masks and error flags as decode_generic: the rows of a
// request's beams in order (row rho: beam rho / (T G), query (rho / G) % T, head
// rho % G), the keys of a workgroup its request's prefix, then the suffixes of
// its rows' beams one after another.
template <int DT, bool SOFTCAP>
__global__ __launch_bounds__(R5_THREADS) void decode_row512(DecodeArgs a, int units, int chunks) {
  kernarg_lines<kernarg_line_count<DecodeArgs>(8)>();
  using E = Elem<DT>;
  using S = typename E::storage;
  using M = Row512<DT>;
  constexpr int PER = M::PER;
  constexpr int D = 32 * PER;
  constexpr int REGION = r5_region<PER>();
  __shared__ __attribute__((aligned(16))) uint8_t tiles[R5_WAVES * REGION];
  __shared__ int64_t t_off[R5_WAVES][2][R5_KEYS];  // per tile key: element offset of its row, -1: none
  __shared__ int t_beam[R5_WAVES][2][R5_KEYS];     // ... its chunk beam; -1: a prefix key, -2: no key
  __shared__ int t_pos[R5_WAVES][2][R5_KEYS];      // ... index in the beam's suffix
  __shared__ int c_len[R5_ROWS], c_s0[R5_ROWS], c_cum[R5_ROWS + 1];
  __shared__ float w_m[R5_WAVES][R5_ROWS], w_l[R5_WAVES][R5_ROWS];

  // workgroup -> (request, KV head, row chunk); blockIdx % 8 is the XCD
  const int seq = blockIdx.x >> 3;
  const int unit = (seq / chunks) * 8 + (blockIdx.x & 7), chunk = seq % chunks;
  if (unit >= units) return;
  const int r = unit / a.Hkv, hk = unit % a.Hkv;
  const int t = threadIdx.x, lane = t & 63, m16 = lane & 15, qd = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int G = a.Hq / a.Hkv, TG = a.T * G;
  const int row0 = chunk * R5_ROWS;
  const int pre_cap = a.prefix_bt_stride * a.bs;
  const int nb0 = a.beam_start[r];
  const int W = a.beam_start[r + 1] - nb0;
  const int P = a.prefix_len[r];
  __asm__ volatile("" ::"s"(P));  // read with the beam range, not after its checks
  if (nb0 < 0 || W < 0 || nb0 + W > a.num_beams || W > a.max_beams) {
    if (t == 0 && chunk == 0) flag_status(a.dev_status, GR_DEV_BAD_LENGTH);
    return;
  }
  if (row0 >= W * TG) return;
  const int nrows = min(R5_ROWS, W * TG - row0);
  const int Pc = min(max(P, 0), pre_cap);
  if (t == 0 && chunk == 0 && Pc != P) flag_status(a.dev_status, GR_DEV_BAD_LENGTH);
  const int b_lo = row0 / TG;
  const int nbm = (row0 + nrows - 1) / TG - b_lo + 1;  // beams in the chunk (<= 16)
  // the wave's first tile's block ids where they are the prefix's, and Q, in
  // flight under the suffix lengths' round trip
  const int kk0 = wave * R5_KEYS + lane;
  int blk0 = -1;
  if (lane < R5_KEYS && kk0 < Pc)
    blk0 = a.prefix_bt[(int64_t)r * a.prefix_bt_stride + (a.bs_shift >= 0 ? kk0 >> a.bs_shift : kk0 / a.bs)];
  const uint8_t* zero = reinterpret_cast<const uint8_t*>(g_zero16);
  // this lane's row and its Q: chunks 4 j + g
  const bool row_ok = m16 < nrows;
  const int rho = row0 + (row_ok ? m16 : 0);
  const int my_b = rho / TG - b_lo, my_qi = (rho / G) % a.T, my_g = rho % G;
  const int64_t my_tok = (int64_t)(nb0 + b_lo + my_b) * a.T + my_qi;
  u32x4_t qf[8];
  {
    const uint8_t* qp = static_cast<const uint8_t*>(a.q) +
                        (my_tok * a.q_tok_stride + (int64_t)(hk * G + my_g) * D) * (int)sizeof(S);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      qf[j] = *reinterpret_cast<const u32x4_t*>(row_ok ? qp + (4 * j + qd) * 16 : zero);
  }
  // wave 0: the chunk's beams' suffix lengths and their running sum
  if (wave == 0) {
    int Lc = 0;
    if (lane < nbm) {
      const int n = nb0 + b_lo + lane;
      const int L = a.suffix_len[n], s0 = a.suffix_start ? a.suffix_start[n] : 0;
      const int suf_cap = a.suffix_bt_stride * a.bs;
      Lc = (L < 0 || s0 < 0 || s0 + L > suf_cap) ? 0 : L;
      if (Lc != L) flag_status(a.dev_status, GR_DEV_BAD_LENGTH);
      c_len[lane] = Lc;
      c_s0[lane] = s0;
    }
    const int incl = wave_incl_scan<32>(Lc);
    if (lane < nbm) c_cum[lane + 1] = incl;
    if (lane == 0) c_cum[0] = 0;
  }
  __syncthreads();
  const int total = Pc + c_cum[nbm];
  const int n_tiles = (total + R5_KEYS - 1) / R5_KEYS;

  const uint8_t* kc = static_cast<const uint8_t*>(a.k_cache) + (int64_t)hk * a.kv_head_stride * (int)sizeof(S);
  const uint8_t* vc = static_cast<const uint8_t*>(a.v_cache) + (int64_t)hk * a.kv_head_stride * (int)sizeof(S);

  const int my_last = c_len[my_b] - a.T + my_qi;  // last suffix index the row sees

  // key kk of tile ti (lanes 0 .. 31 one key each): its block id, then its
  // table entries; the id's load is apart from its use so that it can be in
  // flight under other work
  struct KeyRef { int blk, o, beam, pos; };
  auto key_ref = [&](int ti, bool first = false) {
    KeyRef k{-1, 0, -2, 0};
    const int kk = ti * R5_KEYS + lane;
    if (lane < R5_KEYS && kk < total) {
      int pos = kk;
      const int32_t* bt = a.prefix_bt + (int64_t)r * a.prefix_bt_stride;
      k.beam = -1;
      if (kk >= Pc) {  // suffix slot j: beam kb holds slots c_cum[kb] .. c_cum[kb + 1] - 1
        const int j = kk - Pc;
        int kb = 0;
        while (c_cum[kb + 1] <= j) ++kb;
        k.beam = kb;
        k.pos = j - c_cum[kb];
        pos = c_s0[kb] + k.pos;
        bt = a.suffix_bt + (int64_t)(nb0 + b_lo + kb) * a.suffix_bt_stride;
      }
      const int bi = a.bs_shift >= 0 ? pos >> a.bs_shift : pos / a.bs;
      k.o = pos - bi * a.bs;
      k.blk = first && k.beam == -1 ? blk0 : bt[bi];
    }
    return k;
  };
  auto key_store = [&](int buf, const KeyRef& k) {
    if (lane < R5_KEYS) {
      const bool ok = k.blk >= 0 && k.blk < a.num_blocks;
      if (k.beam != -2 && !ok) flag_status(a.dev_status, GR_DEV_BAD_BLOCK);
      t_off[wave][buf][lane] = ok ? (int64_t)k.blk * a.kv_block_stride + (int64_t)k.o * a.kv_tok_stride : -1;
      t_beam[wave][buf][lane] = ok ? k.beam : -2;
      t_pos[wave][buf][lane] = k.pos;
    }
    // other lanes of the wave read these entries: nothing moves across
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  uint8_t* ktile = tiles + wave * REGION;
  // tile rows 2 i, 2 i + 1 by load i: position p of row key holds chunk p ^ (key % 16)
  auto k_load = [&](int buf) {
#pragma unroll
    for (int i = 0; i < R5_KEYS / 2; ++i) {
      const int key = 2 * i + (lane >> 5);
      const int64_t off = t_off[wave][buf][key];
      const uint8_t* src = off < 0 ? zero : kc + off * (int)sizeof(S) + (((lane & 31) ^ (key & 15)) << 4);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                       (__attribute__((address_space(3))) void*)(ktile + i * 1024), 16, 0, 0);
    }
  };

  f4_t o[2][PER];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int e = 0; e < PER; ++e) o[c][e] = f4_t{0.f, 0.f, 0.f, 0.f};
  float mrow = -INFINITY, lsum = 0.f;  // the row's running maximum; this lane's keys' weights

  if (wave < n_tiles) {
    key_store(0, key_ref(wave, true));
    k_load(0);
  }
  int buf = 0;
  for (int ti = wave; ti < n_tiles; ti += R5_WAVES, buf ^= 1) {
    const bool more = ti + R5_WAVES < n_tiles;
    const KeyRef nx = key_ref(more ? ti + R5_WAVES : n_tiles);  // (n_tiles: every key past the end)
    // V rows of this lane's keys: slot 4 kb + r is key 16 kb + 4 g + r
    u32x4_t vf[2][8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int64_t off = t_off[wave][buf][16 * (s >> 2) + 4 * qd + (s & 3)];
#pragma unroll
      for (int c = 0; c < 2; ++c)
        vf[c][s] = *reinterpret_cast<const u32x4_t*>(off < 0 ? zero : vc + off * (int)sizeof(S) + (16 * c + m16) * 16);
    }
    // This tile's K transfers were issued before the V loads above and return
    // in order: with at most those 16 outstanding they are in LDS.  (The wait
    // is written out: the compiler does not order LDS reads after transfers
    // into LDS in every instantiation.)
    fence<WAIT_VM16>();
    f4_t s2[2] = {f4_t{0.f, 0.f, 0.f, 0.f}, f4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int key = 16 * kb + m16;
        const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(ktile + key * R5_BYTES + (((4 * j + qd) ^ m16) << 4));
        s2[kb] = M::qk(kf, qf[j], s2[kb]);
      }
    }
    // every read of this tile has returned before the next tile lands on it;
    // V too is waited for here, not behind the next tile's transfers
    fence<WAIT_ALL>();
    if (more) {
      key_store(buf ^ 1, nx);
      k_load(buf ^ 1);
    }
    // online softmax of the lane's 8 scores (row m16; keys 16 kb + 4 g + r)
    float p[8], mt = -INFINITY;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int key = 16 * (s >> 2) + 4 * qd + (s & 3);
      float x = s2[s >> 2][s & 3] * a.scale;
      if constexpr (SOFTCAP) x = a.softcap * tanhf(x / a.softcap);
      const int kb = t_beam[wave][buf][key], kp = t_pos[wave][buf][key];
      p[s] = (kb == -1) | ((kb == my_b) & (kp <= my_last)) ? x : -INFINITY;
      mt = fmaxf(mt, p[s]);
    }
    mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float mn = fmaxf(mrow, mt);
    if (__ballot(mn > mrow)) {  // some row's maximum moves: rescale (a row whose own stays multiplies by 1)
      const float al = mrow == -INFINITY ? 0.f : expf(mrow - mn);
      lsum *= al;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < PER; ++e)
#pragma unroll
          for (int u = 0; u < 4; ++u) o[c][e][u] *= al;
      mrow = mn;
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      p[s] = p[s] == -INFINITY ? 0.f : expf(p[s] - mrow);
      lsum += p[s];
    }
    if constexpr (M::PSCALE != 1.f) {
#pragma unroll
      for (int s = 0; s < 8; ++s) p[s] *= M::PSCALE;
    }
    bool terms = DT != GR_DTYPE_F32;  // 16-bit MFMAs on three terms of the weights (wave-uniform)
    if constexpr (DT == GR_DTYPE_F16) {
      bool small = false;
#pragma unroll
      for (int s = 0; s < 8; ++s) small |= (p[s] > 0.f) & (p[s] < M::SPLIT_MIN);
      terms = __ballot(small) == 0;
    }
    if constexpr (DT != GR_DTYPE_F32) {
      if (terms) {
        float pt[3][8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          float t[3];
          split_weight<DT>(p[s], t);
#pragma unroll
          for (int i = 0; i < 3; ++i) pt[i][s] = t[i];
        }
        const u32x4_t pp[3] = {M::pack(pt[0]), M::pack(pt[1]), M::pack(pt[2])};
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int w = 0; w < 4; ++w) {  // dims 2 w, 2 w + 1 of the chunk over the 8 keys
            u32x4_t v0, v1;
#pragma unroll
            for (int h = 0; h < 4; ++h) {
              v0[h] = __builtin_amdgcn_perm(vf[c][2 * h + 1][w], vf[c][2 * h][w], 0x05040100u);
              v1[h] = __builtin_amdgcn_perm(vf[c][2 * h + 1][w], vf[c][2 * h][w], 0x07060302u);
            }
#pragma unroll
            for (int i = 2; i >= 0; --i) {  // the small terms first
              o[c][2 * w] = M::mma(v0, pp[i], o[c][2 * w]);
              o[c][2 * w + 1] = M::mma(v1, pp[i], o[c][2 * w + 1]);
            }
          }
      }
    }
    if constexpr (DT != GR_DTYPE_BF16) {
      if (!terms) {
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int e = 0; e < PER; ++e)
              o[c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(M::v_elem(vf[c][s], e), p[s], o[c][e], 0, 0, 0);
      }
    }
  }

  // ---- merge of the waves' states, in LDS ------------------------------------
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (qd == 0) {
    w_m[wave][m16] = mrow;
    w_l[wave][m16] = lsum;
  }
  __syncthreads();
  // a sink joins the row's softmax: in the maximum and, once, in the sum
  auto row_max = [&](int row, float sink) {
    float m = sink;
#pragma unroll
    for (int w = 0; w < R5_WAVES; ++w) m = fmaxf(m, w_m[w][row]);
    return m;
  };
  {
    const float sink = a.sinks ? a.sinks[hk * G + my_g] : -INFINITY;
    const float m = row_max(m16, sink);
    const float f = mrow == -INFINITY ? 0.f : expf(mrow - m);
    // accumulator (c, e), register u of quarter g: dim PER (16 c + 4 g + u) + e
    float* po = reinterpret_cast<float*>(tiles + wave * REGION) + m16 * r5_pitch<PER>();
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < PER; e += 4)
          *reinterpret_cast<f4_t*>(po + PER * (16 * c + 4 * qd + u) + e) =
              f4_t{o[c][e][u] * f, o[c][e + 1][u] * f, o[c][e + 2][u] * f, o[c][e + 3][u] * f};
  }
  __syncthreads();
  // one thread per (row, 16-byte chunk of the output)
  const int orow = t >> 5, och = t & 31;
  static_assert(R5_ROWS * 32 == R5_THREADS, "a thread per output chunk");
  if (orow >= nrows) return;
  const int orho = row0 + orow;
  // (fp16, whose loop fills the registers: opaque copies, so that the prologue's
  // reciprocals are not spilled across the loop for these quotients)
  int oG = G, oT = a.T;
  if constexpr (DT == GR_DTYPE_F16) __asm__ volatile("" : "+s"(oG), "+s"(oT));
  const int og = orho % oG;
  const int64_t otok = (int64_t)(nb0 + orho / (oT * oG)) * oT + (orho / oG) % oT;
  const float sink = a.sinks ? a.sinks[hk * G + og] : -INFINITY;
  const float m = row_max(orow, sink);
  float l = 0.f;
#pragma unroll
  for (int w = 0; w < R5_WAVES; ++w) {
    const float mw = w_m[w][orow];
    if (mw != -INFINITY) l += w_l[w][orow] * expf(mw - m);
  }
  if (sink != -INFINITY) l += expf(sink - m);
  float v[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) v[e] = 0.f;
#pragma unroll
  for (int w = 0; w < R5_WAVES; ++w) {
    const float* po = reinterpret_cast<const float*>(tiles + w * REGION) + orow * r5_pitch<PER>() + PER * och;
#pragma unroll
    for (int e = 0; e < PER; e += 4) {
      const f4_t x = *reinterpret_cast<const f4_t*>(po + e);
#pragma unroll
      for (int u = 0; u < 4; ++u) v[e + u] += x[u];
    }
  }
#pragma unroll
  for (int e = 0; e < PER; ++e) v[e] = l > 0.f ? v[e] * (1.f / M::PSCALE) / l : 0.f;
  *reinterpret_cast<u32x4_t*>(static_cast<S*>(a.out) + otok * a.out_tok_stride + (int64_t)(hk * G + og) * D + PER * och) =
      M::pack(v);
  if (a.lse_out && och == 0) a.lse_out[otok * a.Hq + hk * G + og] = l > 0.f ? m + logf(l) : -INFINITY;
}

}  // namespace

// Plain, soft-capped and sink decodes whose rows are 512 bytes and 16-byte
// aligned throughout (bases and strides in whole chunks).  Windows, ALiBi and
// fp8 caches stay on the generic kernel.
bool row512_decode_supported(const DecodeArgs& a) {
  const int es = dtype_size(a.dtype);
  if (a.D * es != R5_BYTES || a.kv8 || a.alibi || a.win_left >= 0 || a.win_right >= 0 || !a.causal) return false;
  if (a.num_blocks < 1) return false;
  auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (!al(a.q) || !al(a.out) || !al(a.k_cache) || !al(a.v_cache)) return false;
  const int ch = 16 / es;
  if (a.q_tok_stride % ch || a.out_tok_stride % ch || a.kv_block_stride % ch || a.kv_tok_stride % ch ||
      a.kv_head_stride % ch)
    return false;
  return true;
}

gr_status_t launch_row512_decode(const DecodeArgs& a, hipStream_t stream) {
  const int64_t rows = (int64_t)a.max_beams * a.T * (a.Hq / a.Hkv);
  const int64_t ch64 = (rows + R5_ROWS - 1) / R5_ROWS;
  const int64_t units64 = (int64_t)a.num_reqs * a.Hkv;
  if (ch64 == 0 || units64 == 0) return GR_OK;
  const int64_t nwg = (units64 + 7) / 8 * 8 * ch64;
  if (nwg > 0x7fffffff) return GR_ERR_INVALID_ARG;
  const int units = (int)units64, chunks = (int)ch64;
  const dim3 grid((unsigned)nwg), blk(R5_THREADS);
  const bool cap = a.softcap > 0.f;
#define GR_ROW512(DT)                                                                                       \
  do {                                                                                                      \
    if (cap) hipLaunchKernelGGL((decode_row512<DT, true>), grid, blk, 0, stream, a, units, chunks);         \
    else hipLaunchKernelGGL((decode_row512<DT, false>), grid, blk, 0, stream, a, units, chunks);            \
  } while (0)
  if (a.dtype == GR_DTYPE_F32) GR_ROW512(GR_DTYPE_F32);
  else if (a.dtype == GR_DTYPE_F16) GR_ROW512(GR_DTYPE_F16);
  else GR_ROW512(GR_DTYPE_BF16);
#undef GR_ROW512
  return launch_status();
}

}  // namespace gr
