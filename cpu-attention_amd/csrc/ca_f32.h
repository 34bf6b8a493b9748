// fp32 prefill on the fp16 matrix instructions (included by ca_flash.hip).
//
// The 32-bit MFMA (32x32x2: 64 cycles per 4 KFLOP) bounds fp32 attention at 157 TFLOP/s
// and sums 128 terms of a logit one pair at a time.  Here every fp32 operand x is split
// into two fp16 values, high = fp16(x) and low = fp16(x - high), which hold 23 of its 24
// significant bits (24 where the low one needs at most 11), and a product takes three
// 32x32x16 fp16 MFMAs with fp32 sums: high.high + high.low + low.high (the low.low term
// is below 2^-22 of the product, 2^-25 on average).  That is 96 instead of 512 cycles.
// Probabilities, their sums and the output stay fp32; P is split in the same way for P.V.
//
// Precision.  Against 64 bits the split kernel is closer than the 32-bit MFMAs, whose
// long chains of sums cost more than the splits (2-norm errors, N(0, 1) inputs, before
// -> now): N=1 L=S=2048 H=32 E=128 causal 4.6e-7 -> 2.7e-7, L=S=4096 non-causal 1.2e-6
// -> 7.7e-7, L=S=1024 H=16 E=64 causal 2.8e-7 -> 2.3e-7; with q 8 times larger (peaked
// rows) 1.6e-6 -> 6.9e-7, 2.0e-6 -> 9.3e-7, 1.0e-6 -> 5.0e-7; with lognormal V 4.8e-7 ->
// 1.6e-7, 9.5e-7 -> 6.0e-7, 1.7e-7 -> 1.2e-7.  Over few keys the chains are short and
// the splits would lose up to 45 % (E=64 L=S=17 causal 1.2e-7 -> 1.7e-7): f32_exact
// leaves those calls to the 32-bit MFMAs (E=64 causal up to 56 keys: N=8 H=16 L=S=48 9.6
// us there, 8.5 here; N=16 H=32 L=S=56 14.8, 11.3).
//
// Range.  fp16 reaches from 2^-24 to 65504, so the operands are scaled by powers of two:
// each Q row by its own maximum, K and V by that of the range's first tile, to [2^10,
// 2^11); p by 2^10 (2^14 between two refreshes of the running max).  Called q', k', v'
// and p' then.  Below 2^-2 the low half is subnormal: an operand is off by up to a
// quantum, 2^-25 (2^-25.8 rms), whatever its own size.  What that does to a row is
// compared with what the row came out as, and a query block where it could cost more than
// the 32-bit sums do is redone with the 32-bit MFMAs (ca_f32_pass.inc):
//   logits  are off by c 2^-25.8 (|q'| + |k'|) in 2-norms, at most c 2^-21.3 times the
//           larger of 2^11 and the largest |k'|; allowed is 2^-22.3, or X / 2 times that
//           (a logit of X, in log2 units, is itself rounded by up to 2^-24 X): kF32Logit.
//   O       is off in a row by 2^-25.8 times the root of sum p'^2 (V's quanta, in each
//           dim) and by as much of the root of sum v'^2 (P's quanta, over all dims).  Its
//           largest |O| has to be 2^23.8 times the first (sum p'^2 <= 2^14 sum p') and
//           2^22.8 times the second: kF32RowSum, kF32RowKeys.  So rows whose weight lies
//           on keys of much smaller values, or of none, are redone.
//   columns of V must not hide behind larger ones: in every tile (of kF32TileKeys or more
//           keys), of the 8 keys that a wave stages, one reaches 2^-3 (kF32Dense) in each
//           column, whose quanta then stay below 2^-21.3 of it.  Columns that are 0 in the
//           first tile must be 0 in all (padded head dims), and 8 keys of zeros pass
//           (padded keys).  A column of zeros in some tiles only (a one-hot V, say) is
//           redone: where the others have none, it consists of P's small values, which
//           are quanta themselves.
// (A single value far below both its row's and its column's others keeps its quantum's
// error, small against theirs.)
//   others: a K or V first tile of zeros or of too few keys, a maximum outside 2^-40 ..
//           2^40, a later tile's past 2^5 times the first's, inf or NaN.
// What the first tile shows costs that tile alone (E=64 L=1024 S=8192 H=8, a V channel 1e4
// times the others: 165 us, N(0, 1) 85, 32-bit MFMAs 156), the rest the walk.  Channels of
// K 20 or of V 100 times the others, q 30 times larger or one value of 300 stay on the
// split operands.  The checks cost 0 to 4 % (N=1 L=S=2048 H=32 E=128 causal 147.0 -> 147.8
// us, N=8 L=S=512 H=16 E=64 35.7 -> 37.1, N=1 L=17 S=4096 H=8 E=128 27.6 -> 28.8; N=2
// L=S=17 H=16 E=128 8.2 -> 8.6).
//
// Key groups (KG = 2): a second set of 4 waves on the same rows walks every other tile
// and merges in LDS, as in flash_duo_kernel, for grids that give a CU one block: the
// waves of one block do not cover each other's softmax and splitting (N=1 L=S=2048 H=32
// E=128 causal, 256 pairs: 171 -> 139 us; L=S=4096 H=16 E=64 196 -> 146 us).
//
// Bound: the three MFMAs per product and the splitting of K and V tiles by every block
// of 128 rows.  Measured back to back, 32-bit MFMAs -> now: N=1 L=S=2048 H=32 E=128
// causal 330 -> 139 us (248 TFLOP/s), N=1 L=S=4096 non-causal 2077 -> 909 us (303
// TFLOP/s), N=4 L=S=4096 H=32 E=64 causal 2244 -> 1099 us, N=8 L=S=512 H=16 E=64 81 -> 42
// us, N=1 L=64 S=4096 H=8 E=64 29 -> 21 us.
#pragma once

namespace ca {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
typedef __attribute__((address_space(3))) f16x8 lds_f16x8;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4v;
typedef __attribute__((address_space(3))) s16x4v lds_s16x4;

template <int E>
struct F32Cfg {
  static constexpr int BN = 32;           // keys per tile
  static constexpr int PL = BN * E * 2;   // bytes of one plane (high or low halves) of a tile
  static constexpr int TB = 4 * PL;       // K high, K low, V high, V low
  static constexpr int CH = FlashF32Cfg<E>::CH;
  // Two tile buffers per key group, at least the 32-bit pass's buffers; after them a
  // key group's exchange words: per wave the first tile's largest K and V magnitudes and
  // the columns that its V rows are not all 0 in.
  static constexpr int tiles(int kg) { return 2 * kg * TB > FlashF32Cfg<E>::LDS_BYTES ? 2 * kg * TB : FlashF32Cfg<E>::LDS_BYTES; }
  static constexpr int XW = 8;  // words per wave
  static constexpr int lds_bytes(int kg) { return tiles(kg) + kg * 4 * XW * 4; }
  static constexpr int MERGE = E * 128 + 512;  // a wave's O, m and l for the merge of two groups
  static_assert(4 * MERGE <= tiles(2), "the merge fits the tile buffers");
};

__device__ __forceinline__ uint32_t f16_bits(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }
// The wave's combination of x in every lane: within rows of 16 lanes by rotations (no LDS
// round trips, as shuffles take), then of the 4 rows.
template <typename F>
__device__ __forceinline__ uint32_t wave_fold(uint32_t x, F&& f) {
  x = f(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xf, 0xf, false));  // row_ror:8
  x = f(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x124, 0xf, 0xf, false));
  x = f(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x122, 0xf, 0xf, false));
  x = f(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x121, 0xf, 0xf, false));
  return f(f((uint32_t)__builtin_amdgcn_readlane((int)x, 0), (uint32_t)__builtin_amdgcn_readlane((int)x, 16)),
           f((uint32_t)__builtin_amdgcn_readlane((int)x, 32), (uint32_t)__builtin_amdgcn_readlane((int)x, 48)));
}
__device__ __forceinline__ uint32_t wave_umax(uint32_t x) { return wave_fold(x, umax); }
__device__ __forceinline__ float wave_fsum(float x) {
  return __uint_as_float(wave_fold(__float_as_uint(x), [](uint32_t a, uint32_t b) __attribute__((always_inline)) {
    return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
  }));
}
// a and b, each as two fp16 values high + low (rounded to nearest even).
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  const f16x2 h = {static_cast<_Float16>(a), static_cast<_Float16>(b)};
  hi = f16_bits(h);
  lo = f16_bits(f16x2{static_cast<_Float16>(a - static_cast<float>(h.x)), static_cast<_Float16>(b - static_cast<float>(h.y))});
}

// The larger magnitude of each half of two fp16 pairs (as bits: inf and NaN are largest).
__device__ __forceinline__ uint32_t max_abs16(uint32_t top, uint32_t x) {
  typedef __attribute__((ext_vector_type(2))) unsigned short u16x2;
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, top),
                                                                __builtin_bit_cast(u16x2, x & 0x7fff7fffu)));
}

// The exponent of a finite nonzero |x| = 2^e * [1, 2), as bits; 0 for 0.
__device__ __forceinline__ int exp_of(float mx) { return (int)((__float_as_uint(mx) >> 23) & 255) - 127; }

constexpr int kF32Top = 10;  // the scaled block maximum lies in [2^10, 2^11)

// The power of two that scales values up to mx to kF32Top; not ok: mx is 0, or outside
// 2^-40 .. 2^40 (or inf or NaN).
__device__ __forceinline__ float f32_scale(float mx, bool& ok) {
  const int e = exp_of(mx);
  ok = e >= -40 && e <= 40;
  return ok ? __uint_as_float((uint32_t)(127 + kF32Top - e) << 23) : 1.f;
}

// The limits of the quanta's part of the error (see Range above).
constexpr float kF32Logit = 0.5f;       // c times the larger of 2^11 and the largest |k'|
constexpr float kF32RowKeys = 1.f / 64;  // of the sum of all v' squared
constexpr float kF32RowSum = 1024.f;    // of the sum of p'
constexpr uint32_t kF32Dense = 0x3000;  // fp16 2^-3
// p' = 2^(s c - m) is at most 2^10 at a refresh of m and 2^14 before the next.
constexpr float kF32Lift = 10.f, kF32Slack = 4.f;

// A wave's ballot over its staged chunks, one bit per 4 columns: lanes E / 4 apart hold
// the same columns.
template <int E>
struct F32Cols {
  static constexpr uint32_t ALL = E == 128 ? 0xffffffffu : (1u << (E / 4)) - 1;
  __device__ __forceinline__ static uint32_t of(bool x) {
    const uint64_t b = __ballot(x);
    uint32_t r = (uint32_t)b | (uint32_t)(b >> 32);
    if (E <= 64) r |= r >> 16;
    if (E <= 32) r |= r >> 8;
    return r & ALL;
  }
};

// Keys that a tile needs for a look at V's columns: 4 or more of them lie in every wave's
// rows then, at E = 32 in whole tiles alone.
template <int E>
constexpr int kF32TileKeys = E == 32 ? 32 : 16;

// Calls of few keys stay on the 32-bit MFMAs, which are closer to 64 bits there (N(0, 1),
// L=S: E=32 causal 160 keys 1.85e-7 against 1.9e-7 and more, 193 even, non-causal 48 keys
// 2.17e-7 against 2.20e-7, 64 2.35e-7 against 2.30e-7; E=64 causal 48 keys 1.69e-7 against
// 1.72e-7, 64 1.81e-7 against 1.78e-7, non-causal from 33 keys 2.46e-7 against 2.15e-7)
// and up to 32 keys no slower (E=32 L=S=17 4.5 against 5.4 us), as do calls of too few
// keys for a tile.
inline bool f32_exact(int E, bool causal, int64_t seq_k) {
  if (E == 32) return seq_k <= (causal ? 192 : 56);
  if (E == 64) return seq_k <= (causal ? 56 : 32);
  return seq_k < kF32TileKeys<128>;
}

template <int E, int KG, bool SPLIT>
__global__ __launch_bounds__(256 * KG, 2) void flash_f32_kernel(FlashParams p, int pair) {
  using C = F32Cfg<E>;
  constexpr int BN = C::BN, PL = C::PL, TB = C::TB, CH = C::CH, NS = E / 16, ND = E / 32;
  extern __shared__ __attribute__((aligned(1024))) char f32_smem[];
  static_assert(KG == 1 || !SPLIT, "split calls have one key group");
  const int tid = threadIdx.x & 255, lane = tid & 63;  // thread of its key group
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
  const int li = lane & 31, hf = lane >> 5;
  PairWork pw{};
  if (pair) pw = pair_work(p, kBM, false, blockIdx.x);
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((const lds_void*)f32_smem) + grp * 2 * TB;
  const int sp = SPLIT ? (int)blockIdx.y : 0, splits = SPLIT ? (int)gridDim.y : 1;
  // LDS address of this thread's first staged chunk (8 bytes of halfs): K and V rows,
  // swizzled as the bf16 tiles; chunk i lies RI rows further (at E = 128 every other
  // one with another K swizzle).
  constexpr int RI = 1024 / E;
  const int cr = tid / (E / 4), c4 = tid % (E / 4), col = c4 >> 1;
  const uint32_t kst = lds0 + cr * 2 * E + ((col ^ duo_k_swz<E>(cr)) << 4) + (c4 & 1) * 8;
  const uint32_t vst = lds0 + 2 * PL + cr * 2 * E + ((((col >> 2) ^ duo_v_swz<E>(cr)) << 2 | (col & 3)) << 4) + (c4 & 1) * 8;
  const uint32_t kl = lds0 + li * 2 * E + ((hf ^ duo_k_swz<E>(li)) << 4);
  const int j = lane & 15, dh = (lane >> 4) & 1;
  uint32_t va[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
    va[d] = lds0 + 2 * PL + (4 * hf + (j >> 2)) * 2 * E + ((d ^ duo_v_swz<E>(j >> 2)) << 6) + dh * 32 + (j & 3) * 8;

  const int np = pair ? pw.n : 1;
  uint32_t failed = 0;  // passes whose values the split operands do not hold
#pragma unroll 1
  for (int pass = 0; pass < np; ++pass) {
    if (pass > 0) __syncthreads();  // the tile buffers of the pass before are free
    const BlockWork bw = pair ? BlockWork{pw.b, pw.h, (pass ? pw.qb1 : pw.qb0) * kBM} : block_work(p, blockIdx.x);
    const int L = (int)p.seq_q, S = (int)p.seq_k, diag = S - L;
    const float* qg = reinterpret_cast<const float*>(p.q) + bw.b * p.qs[0] + bw.h * p.qs[2];
    const float* kg = reinterpret_cast<const float*>(p.k) + bw.b * p.ks[0] + bw.h * p.ks[2];
    const float* vg = reinterpret_cast<const float*>(p.v) + bw.b * p.vs[0] + bw.h * p.vs[2];
    const int r0 = (int)bw.q0 + 32 * wv, row = r0 + li;
    const F32Keys kr = f32_keys(p, bw.q0, SPLIT, sp, splits);
    // Group g takes tiles g, g + KG, ...: its round t is tile t KG + g.
    int nkt = (kr.nkt + KG - 1) / KG;
    const int kbeg = (int)kr.kbeg;
    const int kend_w = p.causal ? imin(S, r0 + 32 + diag) : S;

    // Tiles: global -> registers (buffer loads rebased at each tile, zeros past the
    // last key), split into LDS planes by store_one.
    u32x4 reg[CH];
    const int koff = f32_tile_offset<E>(tid, 0, p.ks[1]), voff = f32_tile_offset<E>(tid, 0, p.vs[1]);
    const int kstep = (int)(RI * p.ks[1] * 4), vstep = (int)(RI * p.vs[1] * 4);
    auto load_one = [&](const float* g, int64_t stride, int off, int step, int t, u32x4 (&x)[CH]) __attribute__((always_inline)) {
      const int64_t k0 = kbeg + ((int64_t)t * KG + grp) * BN;
      const __amdgpu_buffer_rsrc_t rs = tile_rsrc(g + k0 * stride, f32_tile_bytes<E>(S, k0, stride));
      asm volatile("" : "+v"(off));  // the chunks' offsets are added here, not kept
#pragma unroll
      for (int i = 0; i < CH; ++i) x[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, off + i * step, 0, 0);
    };
    auto load_k = [&](int t, u32x4 (&x)[CH]) __attribute__((always_inline)) { load_one(kg, p.ks[1], koff, kstep, t, x); };
    auto load_v = [&](int t, u32x4 (&x)[CH]) __attribute__((always_inline)) { load_one(vg, p.vs[1], voff, vstep, t, x); };
    // Not ok: the split operands do not serve the query block (Range, above).
    auto judged = [&](int t) __attribute__((always_inline)) { return S - (kbeg + (t * KG + grp) * BN) >= kF32TileKeys<E>; };
    bool ok = nkt == 0 || judged(0);
    float sk = 1.f, sv = 1.f;
    uint32_t* xw = reinterpret_cast<uint32_t*>(f32_smem + C::tiles(KG)) + grp * 4 * C::XW;
    bool zeros = false;  // some columns of the first V tile are all 0
    uint32_t ktop = 0;   // this thread's largest |k'| (fp16 pairs; inf and NaN are largest)
    float vsum = 0.f;    // per tile and column, its largest v' squared (CH times this bounds the sum)
    // Whether some wave of the block has found the operands not to serve (word 6 or 7).
    auto failing = [&](int word) __attribute__((always_inline)) {
      const bool mine = __any(!ok);
      if (lane == 0) xw[wv * C::XW + word] = mine;
      __syncthreads();
      const uint32_t* all = reinterpret_cast<const uint32_t*>(f32_smem + C::tiles(KG));
      uint32_t any = 0;
#pragma unroll
      for (int w = 0; w < 4 * KG; ++w) any |= all[w * C::XW + word];
      return __builtin_amdgcn_readfirstlane((int)any) != 0;
    };
    // Splits this thread's staged values into the planes of a tile buffer; the largest
    // magnitudes of the high halves of columns 0 and 1 (top.x) and 2 and 3 (top.y).
    auto store_one = [&](const u32x4 (&x)[CH], float sc, uint32_t at0, bool k) __attribute__((always_inline)) {
      u32x2 top = {0, 0};
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        u32x2 hi, lo;
        uint32_t h, l;
        split2(__uint_as_float(x[i].x) * sc, __uint_as_float(x[i].y) * sc, h, l);
        hi.x = h;
        lo.x = l;
        split2(__uint_as_float(x[i].z) * sc, __uint_as_float(x[i].w) * sc, h, l);
        hi.y = h;
        lo.y = l;
        const uint32_t at = (k && E == 128 && (i & 1) ? at0 ^ 128u : at0) + i * RI * 2 * E;
        *(lds_u32x2*)(uintptr_t)at = hi;
        *(lds_u32x2*)(uintptr_t)(at + PL) = lo;
        const uint32_t h0 = hi.x, h1 = hi.y;
        top = u32x2{max_abs16(top.x, h0), max_abs16(top.y, h1)};
      }
      return top;
    };
    auto store_k = [&](const u32x4 (&x)[CH], int buf) __attribute__((always_inline)) {
      const u32x2 top = store_one(x, sk, kst + buf * TB, true);
      ktop = max_abs16(max_abs16(ktop, top.x), top.y);
    };
    // The columns of V tile t that the wave's 8 rows hold a nonzero value in.
    auto held = [&](const u32x4 (&x)[CH], uint32_t (&n)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t bits = 0;
#pragma unroll
        for (int i = 0; i < CH; ++i) bits |= x[i][j];
        n[j] = F32Cols<E>::of((bits & 0x7fffffffu) != 0);
      }
    };
    auto store_v = [&](const u32x4 (&x)[CH], int t) __attribute__((always_inline)) {
      const u32x2 top = store_one(x, sv, vst + (t & 1) * TB, false);
      const uint32_t t0 = top.x, t1 = top.y;
      vsum = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, t0), __builtin_bit_cast(f16x2, t0), vsum, false);
      vsum = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, t1), __builtin_bit_cast(f16x2, t1), vsum, false);
      if (!judged(t)) return;
      const uint32_t r[4] = {F32Cols<E>::of((top.x & 0xffff) >= kF32Dense), F32Cols<E>::of((top.x >> 16) >= kF32Dense),
                             F32Cols<E>::of((top.y & 0xffff) >= kF32Dense), F32Cols<E>::of((top.y >> 16) >= kF32Dense)};
      if (__builtin_expect((r[0] & r[1] & r[2] & r[3]) == F32Cols<E>::ALL && !zeros, 1)) return;
      uint32_t n[4];
      held(x, n);
      if ((n[0] | n[1] | n[2] | n[3]) == 0) return;  // 8 rows of zeros
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t first = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) first |= xw[w * C::XW + 2 + j];
        ok &= (((first & ~r[j]) | (n[j] & ~first)) & F32Cols<E>::ALL) == 0;
      }
    };

    u32x4 vreg0[CH];
    if (nkt > 0) {
      load_k(0, reg);
      load_v(0, vreg0);
    }
    // Q, scaled per row: lane (row li, half hf) holds dims 16 s + 8 hf .. +7.
    f16x8 qh[NS], ql[NS];
    float c = 0.f;
    {
      float qv[NS][8];
      uint32_t mb = 0;  // the row's largest magnitude, as bits (inf and NaN are largest)
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          u32x4 v = {0, 0, 0, 0};
          if (row < L) v = *reinterpret_cast<const u32x4*>(qg + (int64_t)row * p.qs[1] + 16 * s + 8 * hf + 4 * u);
          const float f[4] = {__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w)};
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            qv[s][4 * u + x] = f[x];
            mb = umax(mb, __float_as_uint(f[x]) & 0x7fffffffu);
          }
        }
      const float mx = __uint_as_float(umax(mb, __shfl_xor(mb, 32)));
      bool fits;
      // A negative softmax scale turns Q's sign instead, and a zero one zeroes Q, so
      // that c > 0: the running max is taken of the raw logits, and -inf * c is -inf.
      float sq = f32_scale(mx, fits);
      ok &= __all(fits || mx == 0.f);
      c = fabsf(p.c) / sq;
      sq = p.c < 0.f ? -sq : sq;
      if (p.c == 0.f || mx == 0.f) {  // logits of 0 for any small c > 0
        sq = 0.f;
        c = 0x1p-60f;
      }
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        u32x4 h, l;
        uint32_t a, b;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          split2(qv[s][2 * x] * sq, qv[s][2 * x + 1] * sq, a, b);
          h[x] = a;
          l[x] = b;
        }
        qh[s] = __builtin_bit_cast(f16x8, h);
        ql[s] = __builtin_bit_cast(f16x8, l);
      }
    }
    // The block's K and V scales, from its first tile.
    if (nkt > 0) {
      uint32_t mk = 0, mv = 0;
#pragma unroll
      for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const uint32_t a = reg[i][x] & 0x7fffffffu, b = vreg0[i][x] & 0x7fffffffu;
          mk = umax(mk, a);
          mv = umax(mv, b);
        }
      mk = wave_umax(mk);
      mv = wave_umax(mv);
      uint32_t n[4];
      held(vreg0, n);
      if (lane == 0) {
        uint32_t* w = xw + wv * C::XW;
        w[0] = mk;
        w[1] = mv;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[2 + j] = n[j];
      }
      __syncthreads();
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        mk = umax(mk, xw[x * C::XW]);
        mv = umax(mv, xw[x * C::XW + 1]);
#pragma unroll
        for (int j = 0; j < 4; ++j) n[j] |= xw[x * C::XW + 2 + j];
      }
      zeros = __any((n[0] & n[1] & n[2] & n[3]) != F32Cols<E>::ALL);
      bool fk, fv;
      sk = f32_scale(__uint_as_float(mk), fk);
      sv = f32_scale(__uint_as_float(mv), fv);
      c /= sk;
      ok &= fk && fv;
      store_k(reg, 0);
      store_v(vreg0, 0);
      if (failing(6)) nkt = 0;  // the 32-bit pass without the walk first
    }

    f32x16 o[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) o[d] = f32x16{};
    // m: the running max in scaled log2 units less kF32Lift.
    float m = -INFINITY, l = 0.f;
    for (int t = 0; t < nkt; ++t) {
      const uint32_t buf = (t & 1) * TB;
      load_k(t + 1, reg);  // past the last tile: zeros past S, never used
      const int k0 = kbeg + (t * KG + grp) * BN;
      const bool mine = k0 < kend_w && (KG == 1 || t * KG + grp < kr.nkt);
      f32x16 st = f32x16{}, sx = f32x16{};
      if (mine) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const uint32_t at = (kl + buf) ^ (uint32_t)(s << 5);
          const f16x8 kh = *(lds_f16x8*)(uintptr_t)at, kw = *(lds_f16x8*)(uintptr_t)(at + PL);
          sx = __builtin_amdgcn_mfma_f32_32x32x16_f16(kw, qh[s], sx, 0, 0, 0);
          st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[s], st, 0, 0, 0);
          sx = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[s], sx, 0, 0, 0);
        }
        st += sx;
      }
      if (t + 1 < nkt) store_k(reg, (t & 1) ^ 1);
      load_v(t + 1, reg);
      if (mine) {
        if (k0 + BN > S || (p.causal && k0 + BN - 1 > r0 + diag)) {
          int vis = S - 1 - k0;
          if (p.causal) vis = imin(vis, row + diag - k0);
          vis -= 4 * hf;
          asm volatile("" : "+v"(vis));
#pragma unroll
          for (int r = 0; r < 16; ++r) st[r] = vis >= 8 * (r >> 2) + (r & 3) ? st[r] : -INFINITY;
        }
        float mt = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) mt = fmaxf(mt, st[r]);
        mt = fmaxf(mt, __shfl_xor(mt, 32)) * c - kF32Lift;
        if (__any(mt > m + kF32Slack)) {
          const float mn = fmaxf(m, mt), alpha = __builtin_amdgcn_exp2f(m - (mn == -INFINITY ? 0.f : mn));
          l *= alpha;
#pragma unroll
          for (int d = 0; d < ND; ++d) o[d] *= alpha;
          m = mn;
        }
        const float nm = m == -INFINITY ? 0.f : -m;
        float ls = 0.f;
        f16x8 ph[2], pl[2];
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
          u32x4 h, w;
          uint32_t a, b;
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const float e0 = __builtin_amdgcn_exp2f(fmaf(st[8 * cc + 2 * x], c, nm));
            const float e1 = __builtin_amdgcn_exp2f(fmaf(st[8 * cc + 2 * x + 1], c, nm));
            ls += e0;
            ls += e1;
            split2(e0, e1, a, b);
            h[x] = a;
            w[x] = b;
          }
          ph[cc] = __builtin_bit_cast(f16x8, h);
          pl[cc] = __builtin_bit_cast(f16x8, w);
        }
        l += ls;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
          for (int d = 0; d < ND; ++d) {
            s16x4v x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
              x[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(va[d] + buf + (u >> 1) * PL + (16 * cc + 8 * (u & 1)) * 2 * E));
            const f16x8 vh = __builtin_bit_cast(f16x8, __builtin_shufflevector(x[0], x[1], 0, 1, 2, 3, 4, 5, 6, 7));
            const f16x8 vw = __builtin_bit_cast(f16x8, __builtin_shufflevector(x[2], x[3], 0, 1, 2, 3, 4, 5, 6, 7));
            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vw, ph[cc], o[d], 0, 0, 0);
            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl[cc], o[d], 0, 0, 0);
            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph[cc], o[d], 0, 0, 0);
          }
      }
      if (t + 1 < nkt) store_v(reg, t + 1);
      __syncthreads();
    }

    {
      // The row's largest |O|, its sum of p', and what all waves staged, against the limits.
      uint32_t kt = wave_umax(umax(ktop & 0xffff, ktop >> 16));
      const float vw = wave_fsum(vsum);
      if (lane == 0) {
        xw[wv * C::XW] = kt;
        xw[wv * C::XW + 1] = __float_as_uint(vw);
      }
      __syncthreads();
      float vs = 0.f, top = 0.f;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        kt = umax(kt, xw[x * C::XW]);
        vs += __uint_as_float(xw[x * C::XW + 1]);
      }
      const float kv = static_cast<float>(__builtin_bit_cast(f16x2, umax(kt, 0x6800u)).x);  // 2^11 or more
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) top = fmaxf(top, fabsf(o[d][r]));
      top = fmaxf(top, __shfl_xor(top, 32));
      const float lt = l + __shfl_xor(l, 32);
      if (row < L && lt != 0.f)
        ok &= kt < 0x7c00u && vs < INFINITY && top * top >= fmaf(lt, kF32RowSum, vs * (CH * kF32RowKeys)) &&
              c * kv <= kF32Logit * fmaxf(1.f, 0.5f * fabsf(m + kF32Lift));
    }
    if (failing(7)) {
      failed |= 1u << pass;
      continue;
    }
    float isv = 1.f / sv;
    if constexpr (KG == 2) {
      // Group 1's sums (in the values' own scale) go through LDS to group 0.
      float* mb = reinterpret_cast<float*>(f32_smem + wv * C::MERGE) + lane;
      if (grp == 1) {
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) mb[64 * (16 * d + r)] = o[d][r] * isv;
        mb[64 * 16 * ND] = m;
        mb[64 * 16 * ND + 64] = l;
      }
      __syncthreads();
      if (grp == 1) continue;
      const float m1 = mb[64 * 16 * ND], mn = fmaxf(m, m1), mu = mn == -INFINITY ? 0.f : mn;
      const float w0 = __builtin_amdgcn_exp2f(m - mu), w1 = __builtin_amdgcn_exp2f(m1 - mu);
      l = l * w0 + mb[64 * 16 * ND + 64] * w1;
      m = mn;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = o[d][r] * (isv * w0) + mb[64 * (16 * d + r)] * w1;
      isv = 1.f;
    }
    const float lt = l + __shfl_xor(l, 32);
    if (row < L) {
      float* po;
      float f;
      if constexpr (SPLIT) {
        const int64_t slot = ((bw.b * p.heads + bw.h) * p.seq_q + row) * splits + sp;
        po = p.part_acc + slot * E;
        f = isv;
        if (hf == 0) {
          p.part_ml[2 * slot] = m;
          p.part_ml[2 * slot + 1] = lt;
        }
      } else {
        po = reinterpret_cast<float*>(p.out) + ((bw.b * p.seq_q + row) * p.heads + bw.h) * E;
        f = lt > 0.f ? isv / lt : 0.f;
      }
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<f32x4*>(po + 32 * d + 8 * g + 4 * hf) =
              f32x4{o[d][4 * g] * f, o[d][4 * g + 1] * f, o[d][4 * g + 2] * f, o[d][4 * g + 3] * f};
    }
  }
  if (grp == 1) return;  // the 32-bit pass takes one group (its barriers wait for the waves still running)
#pragma unroll 1
  for (int pass = 0; pass < np; ++pass) {
    if (!(failed >> pass & 1)) continue;
    __syncthreads();
    const BlockWork bw = pair ? BlockWork{pw.b, pw.h, (pass ? pw.qb1 : pw.qb0) * kBM} : block_work(p, blockIdx.x);
#include "ca_f32_pass.inc"
  }
}

}  // namespace ca
