// bf16 prefill of short and middle key ranges (flash_duo_kernel), included by
// ca_flash.hip, whose tile helpers it uses.
//
// flash_bf16_p64_kernel runs one 64-row wave per SIMD with the whole register file:
// the highest rate on long walks, but nothing covers a wave's waits, its 256-row
// blocks leave CUs idle in small calls, and a pass costs ~12k cycles beside its key
// tiles.  Here a wave holds 32 query rows in at most 256 registers, so two or three
// waves share a SIMD and two or three blocks a CU: one block's first loads, diagonal
// and output overlap another's MFMAs, and a 128-row block splits a call twice as
// finely.  The price is the LDS operand traffic (each K and V^T operand feeds one
// MFMA instead of two).  On long walks that costs power, and so clock: non-causal
// N=4 L=S=4096 H=32 E=128 takes 10 % fewer cycles than on the 64-row kernel (13.6M
// against 15.1M, summed over the XCDs) but at 1.77 instead of 2.04 GHz, and is 4 %
// slower; duo_plan leaves such calls there.
//
//   S^T = K Q^T and O^T += V^T P^T as in the 64-row kernel (32x32x16 MFMAs, a lane
//   owns one query row); the S of tile t + 1, the softmax of tile t and the P.V of
//   tile t form one stream with a fixed order (DuoSeq), the fixed row max and its
//   safe walk are the 64-row kernel's (fix_max).
//
// Key groups (KG = 2): the block has a second set of 4 waves on the same rows; group
// g walks tiles g, g + 2, ... through LDS buffers of its own, and the groups merge in
// LDS at the end.  It halves the serial walk of a call whose blocks do not fill the
// chip, with no partials in memory.  Both groups of a fast walk take p against the max
// fixed at group 0's first tile, the pass's: one walk over all the tiles has that max
// too, so P is rounded as there and the groups' sums add up whatever their sizes.  (A
// max of each group's own can lie 2^126 from the other's while the rows' weight lies
// in the lower one, whose merge weight flushes to 0.)
// Split mode: the keys of each query block over gridDim.y blocks, partials merged by
// the combine kernel (few query blocks over long keys).
// Pairs (causal): query blocks (nqb - 1 - j, j) one after the other, so every block
// walks about the same number of tiles.
#pragma once

namespace ca {

template <int E, int KG>
struct DuoCfg {
  static constexpr int NW = 4;       // waves per key group
  static constexpr int BM = 32 * NW; // query rows per block
  static constexpr int BN = kTileKeys;
  static constexpr int CPR = E / 8;  // 16-byte chunks per row
  static constexpr int TB = BN * E * 2;  // bytes per tile buffer (no padding: swizzled)
  // Two buffers each for K and V: K(t + 2) and V(t + 1) load during tile t.  Three
  // or four of each measured no faster (N=1 L=1536 S=2048 H=20 E=64 25.1, 26.4 us):
  // the walk does not wait for its loads.
  static constexpr int NB = 2;
  static constexpr int GROUP_BYTES = 2 * NB * TB;  // LDS of one key group
  static constexpr int TILES = KG * GROUP_BYTES;
  static constexpr int LDS_BYTES = TILES + (KG == 2 ? 4 * BM : 0);  // the rows' fixed max after the tiles
  static constexpr int NL = BN * CPR / (64 * NW);  // direct loads per thread and tile (K or V)
  static constexpr int STAGE_ROW = 2 * E + 16;     // output staging: bytes per row, padded
  static constexpr int MERGE = E * 128 + 512;      // a wave's O, m and l for the merge of two groups
  // Waves per SIMD the registers must allow: 3 where 168 registers hold a wave.
  static constexpr int WAVES = KG == 1 && E <= 64 ? 3 : 2;
  static_assert(NL * 64 * NW == BN * CPR, "the loads fill a tile exactly");
  static_assert(NW * 32 * STAGE_ROW <= TILES, "the staging fits the tile buffers");
  static_assert(KG == 1 || (NW * MERGE <= TILES && 32 * STAGE_ROW <= MERGE), "the merge fits the tile buffers");
};

// LDS swizzles (tiles are unpadded: a direct load fills 64 consecutive chunks).
// K rows: the chunk column is xored with the row's place so that 16 consecutive
// rows of one column lie in 16 different 16-byte slots of the 256 bytes the
// banks span.  V rows: 64-byte segments are permuted so that 4 consecutive rows
// of one segment lie in 4 different 64-byte slots.
template <int E>
__host__ __device__ inline int duo_k_swz(int row) {
  constexpr int CPR = E / 8, RP = 16 / CPR;
  return (row / RP) & (CPR - 1);
}
template <int E>
__host__ __device__ inline int duo_v_swz(int row) {
  constexpr int NSEG = E / 32, RP = 4 / NSEG;
  return (row / RP) & (NSEG - 1);
}

// Byte offset in the source tile of the 16-byte chunk that lane `lane` of wave wv
// loads into LDS chunk (4 i + wv) * 64 + lane (rows `stride` elements apart).
template <int E, bool V>
__host__ __device__ inline int duo_tile_offset(int wv, int lane, int i, int stride) {
  constexpr int CPR = E / 8;
  const int P = (4 * i + wv) * 64 + lane, r = P / CPR, c = P % CPR;
  const int col = V ? ((((c >> 2) ^ duo_v_swz<E>(r)) << 2) | (c & 3)) : (c ^ duo_k_swz<E>(r));
  return (r * stride + 8 * col) * 2;
}

// A block's work: a (batch, head) and query block qb0, or the causal pair (qb0, qb1).
struct DuoWork {
  uint32_t b, h, qb0, qb1;
  int n;
};
__host__ __device__ inline DuoWork duo_work(const FlashParams& p, int bm, bool pair, uint32_t bid, uint32_t nb) {
  const uint32_t nqb = ((uint32_t)p.seq_q + bm - 1) / bm, heads = (uint32_t)p.heads, per = pair ? (nqb + 1) / 2 : nqb;
  const uint32_t x = bid & 7, px = nb >> 3, rem = nb & 7;
  const uint32_t lg = x * px + (x < rem ? x : rem) + (bid >> 3);  // xcd_remap
  const uint32_t bh = lg / per, j = lg - bh * per;
  DuoWork w;
  w.b = bh / heads;
  w.h = bh - w.b * heads;
  w.qb0 = nqb - 1 - j;
  w.qb1 = j;
  w.n = pair && w.qb0 != j ? 2 : 1;
  return w;
}

// The keys of query block q0 for the wave at rows r0 .. r0 + 31 of key group grp (of
// kg): the pass's keys [kbeg, kbeg + keys) (the split mode's share: whole tiles, empty
// past the pass's last key), nkt rounds of one tile per group for the whole block, of
// which the wave computes nkt_w.
struct DuoKeys {
  int kbeg, keys, nkt, nkt_w;
};
__host__ __device__ inline DuoKeys duo_keys(const FlashParams& p, int q0, int r0, bool split, int sp, int splits, int kg,
                                            int grp) {
  constexpr int BM = DuoCfg<64, 1>::BM, BN = DuoCfg<64, 1>::BN;
  const int L = (int)p.seq_q, S = (int)p.seq_k, diag = S - L;
  int kend = p.causal ? imin(S, q0 + BM + diag) : S;
  DuoKeys k;
  k.kbeg = 0;
  if (split) {
    const int chunk = (int)(((uint32_t)(S + BN - 1) / BN + splits - 1) / splits) * BN;
    k.kbeg = imin(sp * chunk, imax(kend, 0));
    kend = imin(k.kbeg + chunk, kend);
  }
  k.keys = kend - k.kbeg;
  k.nkt = k.keys > 0 ? (k.keys + kg * BN - 1) / (kg * BN) : 0;
  const int kw = (p.causal ? imin(kend, r0 + 32 + diag) : kend) - k.kbeg;
  k.nkt_w = (kw > 0 && r0 < L) ? ((kw + BN - 1) / BN - grp + kg - 1) / kg : 0;
  return k;
}

// The MFMA stream of one key tile (one 32-row column block): S of the next tile
// (2 E / 16 MFMAs) and P.V of this one (4 groups of 16 keys x E / 32), in the order
// in which the operands become ready beside the softmax of this tile.  Score x of the
// lane's 32 is begun in slot sl(x), over about three quarters of the slots, and its P
// is there two slots later; a P.V MFMA goes as soon as its 16 keys' P is complete, the
// S MFMAs fill the other slots.
template <int E>
struct DuoSeq {
  static constexpr int NS2 = 2 * (E / 16), ND = E / 32, NM = NS2 + 4 * ND;
  static constexpr int PN = E == 128 ? 3 : 1, PD = E == 128 ? 4 : (E == 64 ? 3 : 6);
  static constexpr int sl(int x) { return x * PN / PD; }
  static constexpr int MAXS = NM + 16;
  int what[MAXS] = {};  // per slot: -1 nothing, j < NS2 an S MFMA, NS2 + q a P.V MFMA
  int n = 0;
  constexpr DuoSeq() {
    int s = 0, q = 0;
    for (int i = 0; s < NS2 || q < 4 * ND || i < sl(31) + 3; ++i) {
      const bool ready = q < 4 * ND && i >= sl(8 * (q / ND) + 7) + 2;
      what[i] = ready ? NS2 + q++ : (s < NS2 ? s++ : -1);
      n = i + 1;
    }
  }
};

// How a tiled bf16 call runs: kg 0 for flash_bf16_p64_kernel by `tiled`, else the
// duo kernel with kg key groups, splits of its keys (1: none) and causal pairs or not.
//
// With items = batch x heads x ceil(L / 128) blocks and T = ceil(S / 64) key tiles, and
// two resident blocks of one key group per CU (or one of two), measured on MI355X
// back to back, start -> now in us (E = 64 / E = 128):
//   up to 256 items: two key groups past 8 tiles (N=1 L=S=1500 H=20 non-causal 31.7 ->
//     18.5, L=S=2048 H=16 E=128 causal 54.5 -> 31.9; one group 35.3), one up to 8 (N=1
//     L=S=512 H=16 causal 16.3 -> 9.0, L=256 S=512 H=16 E=128 21.4 -> 12.8).
//   257 to 512 items, causal with fewer than twice as many keys as rows: pairs with two groups from 32 tiles (N=1 L=S=4096 H=16
//     74.6 -> 47.8 / 103.3 -> 75.3; pairs with one group 51.5 / 78.5, unpaired 67.0 /
//     99.1), pairs with one group from 12 (L=S=1024 H=48 E=128 33.4 -> 26.1, unpaired
//     29.4), unpaired below (L=S=700 H=60 19.5 -> 13.2 / 25.9 -> 19.6, pairs 15.8 /
//     22.2).  Others: one group (L=S=2048 H=24 40.1 -> 38.1, two groups 43.1).
//   more items, causal: pairs (N=16 L=S=1024 H=32 149 -> 116 / 219 -> 197, unpaired 128 /
//     220); others: one query block per block.
//   up to 64 items from 16 tiles, up to 85 from 32: keys split so that about 256 blocks
//     walk (N=1 L=64 S=8192 H=8 16.8 -> 13.0, L=512 S=4096 H=12 22.8 -> 20.6); from 65
//     items and 96 tiles, or 86 to 170 items from 40 tiles, about 512 (L=512 S=8192 H=20
//     39.5 -> 37.8).  At least 4 tiles per split.  Shorter ones run two groups
//     unsplit: the combine costs ~4 us (L=S=1024 H=16: 13.2, split in 2 20.5).  The
//     workspace is the one the 64-row kernel's split asks for, which is at least as large.
// The 64-row kernel keeps the E = 128 calls it fills whole rounds of the chip with:
// non-causal from 40 tiles (N=4 L=S=4096 H=32: 924 against 962; L=S=2048 H=32 is even,
// and at 384 of its blocks, 1.5 rounds, L=S=4096 H=24 takes 209.6 against 187.0 here),
// causal from 96 (N=1 L=S=8192 H=32 478.7 against 486.0; N=2 L=S=4096 H=32 272 against
// 265); and its split mode at E = 128 from 65 items and 96 tiles (L=512 S=8192 H=40 99.9
// against 101.8).
struct DuoPlan {
  int kg;
  int64_t splits;
  bool pair;
  int64_t gx;
};
inline DuoPlan duo_plan(const FlashParams& p, int E, const FlashPlan& tiled) {
  constexpr int BM = DuoCfg<64, 1>::BM, BN = DuoCfg<64, 1>::BN;
  const int64_t nqb = cdiv(p.seq_q, BM), items = p.batch * p.heads * nqb, T = cdiv(p.seq_k, BN);
  const int64_t items64 = p.batch * p.heads * cdiv(p.seq_q, 256);  // the 64-row kernel's blocks
  const bool tri = p.causal && p.seq_k < 2 * p.seq_q;  // else the blocks' work is nearly even
  DuoPlan d{0, 1, false, items};
  if (items > 0x7fffffff) return d;
  if (E == 128) {
    if (tiled.split && items > 64 && T >= 96) return d;
    if (!tiled.split && tri && items64 > 256 && T >= 96) return d;
    if (!tiled.split && !tri && T >= 40 && 10 * items64 >= 9 * 256 * cdiv(items64, 256)) return d;
  }
  d.kg = 1;
  if (tiled.split && (items <= 64 ? T >= 16 : (items <= 85 ? T >= 32 : items <= 170 && T >= 40))) {
    d.splits = (items > 85 || (items > 64 && T >= 96) ? 512 : 256) / items;
    d.splits = d.splits < T / 4 ? d.splits : T / 4;
    d.splits = d.splits < tiled.splits ? d.splits : tiled.splits;
    if (d.splits > 1) return d;
    d.splits = 1;
  }
  if (items <= 256) {
    d.kg = T > 8 ? 2 : 1;
  } else if (tri) {
    d.kg = items <= 512 && T >= 32 ? 2 : 1;
    d.pair = items > 512 || T >= 12;
  }
  if (d.pair) d.gx = p.batch * p.heads * ((nqb + 1) / 2);
  return d;
}

template <int E, int KG, bool SPLIT>
__global__ __launch_bounds__(256 * KG, (DuoCfg<E, KG>::WAVES)) void flash_duo_kernel(FlashParams p, int pair) {
  static_assert(KG == 1 || !SPLIT, "split calls have one key group");
  using C = DuoCfg<E, KG>;
  constexpr int BM = C::BM, BN = C::BN, NL = C::NL, NB = C::NB, TB = C::TB, NS = E / 16, ND = E / 32, NS2 = 2 * NS;
  extern __shared__ __attribute__((aligned(1024))) char duo_smem[];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, hf = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wv = wid & 3, grp = KG == 1 ? 0 : wid >> 2;  // wave of its key group, key group
  const DuoWork dw = duo_work(p, BM, pair != 0, blockIdx.x, gridDim.x);
  // Positions and token strides fit 32 bits (the plan declines otherwise).
  const int L = (int)p.seq_q, S = (int)p.seq_k, diag = S - L;
  const int qs1 = (int)p.qs[1], ks1 = (int)p.ks[1], vs1 = (int)p.vs[1];
  const uint16_t* qg = reinterpret_cast<const uint16_t*>(p.q) + (int64_t)dw.b * p.qs[0] + (int64_t)dw.h * p.qs[2];
  const uint16_t* kg = reinterpret_cast<const uint16_t*>(p.k) + (int64_t)dw.b * p.ks[0] + (int64_t)dw.h * p.ks[2];
  const uint16_t* vg = reinterpret_cast<const uint16_t*>(p.v) + (int64_t)dw.b * p.vs[0] + (int64_t)dw.h * p.vs[2];
  uint16_t* out = reinterpret_cast<uint16_t*>(p.out) + ((int64_t)dw.b * p.seq_q * p.heads + dw.h) * E;
  int koff[NL], voff[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    koff[i] = duo_tile_offset<E, false>(wv, lane, i, ks1);
    voff[i] = duo_tile_offset<E, true>(wv, lane, i, vs1);
  }
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((const lds_void*)duo_smem) + grp * C::GROUP_BYTES;

  // A stream of tiles into the rotating K or V buffers: the group's next tile through
  // a window cut at the range's last key (empty past it).  The loads are inline
  // assembly, as the 64-row kernel's: loads_landed_barrier waits for them.
  struct Stream {
    uint64_t addr;
    int rows;
    uint32_t buf;
  } ks, vs;
  const uint32_t kbuf0 = lds0 + wv * 1024, vbuf0 = kbuf0 + NB * TB;
  auto issue = [&](Stream& x, uint32_t buf0, int stride2, const int (&off)[NL]) __attribute__((always_inline)) {
    const i32x4 rs = {__builtin_amdgcn_readfirstlane((int)(uint32_t)x.addr),
                      __builtin_amdgcn_readfirstlane((int)((x.addr >> 32) & 0xffff)),
                      __builtin_amdgcn_readfirstlane(tile_window<E>(x.rows, stride2)), 0x00020000};
    const uint32_t base = __builtin_amdgcn_readfirstlane(x.buf);
#pragma unroll
    for (int i = 0; i < NL; ++i)
      asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                   :
                   : "s"(base + i * 4096), "v"(off[i]), "s"(rs)
                   : "memory");
    x.addr += (uint64_t)(uint32_t)(BN * stride2) * KG;
    x.rows -= KG * BN;
    x.buf = x.buf == buf0 ? buf0 + TB : buf0;
  };
  auto issue_k = [&]() __attribute__((always_inline)) { issue(ks, kbuf0, 2 * ks1, koff); };
  auto issue_v = [&]() __attribute__((always_inline)) { issue(vs, vbuf0, 2 * vs1, voff); };

  // K operand: row li (+ 32 kt), chunk 2 s + hf swizzled.  V^T operand: as v_operand.
  const uint32_t kl = lds0 + li * 2 * E + ((hf ^ duo_k_swz<E>(li)) << 4);
  const int j = lane & 15, dh = (lane >> 4) & 1;
  uint32_t va[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
    va[d] = lds0 + NB * TB + (4 * hf + (j >> 2)) * 2 * E + ((d ^ duo_v_swz<E>(j >> 2)) << 6) + dh * 32 + (j & 3) * 8;
  auto kread = [&](uint32_t base, int q) __attribute__((always_inline)) {
    return *(lds_bf16x8*)(uintptr_t)((base ^ (uint32_t)((q >> 1) << 5)) + (q & 1) * 64 * E);
  };
  auto vread = [&](uint32_t off, int q) __attribute__((always_inline)) {
    bf16x4v a[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
      a[u] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
          (lds_bf16x4*)(uintptr_t)(va[q % ND] + off + (16 * (q / ND) + 8 * u) * 2 * E));
    return bf16x8{a[0][0], a[0][1], a[0][2], a[0][3], a[1][0], a[1][1], a[1][2], a[1][3]};
  };

#pragma unroll 1
  for (int pass = 0; pass < dw.n; ++pass) {
    if (pass > 0) __syncthreads();  // every wave is done with the staging of the pass before
    const int q0 = (int)(pass == 0 ? dw.qb0 : dw.qb1) * BM, r0 = q0 + 32 * wv;
    const DuoKeys kr = duo_keys(p, q0, r0, SPLIT, SPLIT ? (int)blockIdx.y : 0, SPLIT ? (int)gridDim.y : 1, KG, grp);
    const int kbeg = kr.kbeg, nkt = kr.nkt, nkt_w = kr.nkt_w;

    bf16x8 qr[NS];  // Q^T as B operands: dims 16 s + 8 hf .. of row r0 + li
    {
      const __amdgpu_buffer_rsrc_t rs = tile_rsrc(qg + (int64_t)r0 * qs1, ((int64_t)(L - 1 - r0) * qs1 + E) * 2);
#pragma unroll
      for (int s = 0; s < NS; ++s)
        qr[s] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, (li * qs1 + 16 * s + 8 * hf) * 2, 0, 0));
    }
    f32x16 o[ND];  // O^T: dims 32 d + 8 (r / 4) + 4 hf + r % 4
    float m, nmu, l;

    // -inf for the keys of tile t (of this group) past the row's limit.
    auto mask = [&](f32x16 (&sx)[2], int t) __attribute__((always_inline)) {
      const int k0 = kbeg + (t * KG + grp) * BN;
      if (k0 + BN > S || (p.causal && k0 + BN - 1 > r0 + diag)) {
        int vis = S - 1 - k0;
        if (p.causal) vis = imin(vis, r0 + li + diag - k0);
        vis -= 4 * hf;
        asm volatile("" : "+v"(vis));  // keeps the compares here (hoisted out of the walk, they spill)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int r = 0; r < 16; ++r) sx[kt][r] = vis >= 32 * kt + 8 * (r >> 2) + (r & 3) ? sx[kt][r] : -INFINITY;
      }
    };
    auto row_max = [&](const f32x16 (&sx)[2]) __attribute__((always_inline)) {
      float mx = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sx[kt][r]);
      return fmaxf(mx, __shfl_xor(mx, 32)) * p.c;
    };

    // One walk over the group's tiles; false: a row's sum of p over a tile passed the
    // fixed max's headroom (or is NaN), see P64Rows::fix_max.  `safe`: with a running
    // max, refreshed when a tile's passes it by 8 log2 units.
    auto walk = [&](const bool safe) __attribute__((always_inline)) {
      constexpr float kHeadSum = 18446744073709551616.f;  // 2^64
      bool fine = true;
#pragma unroll
      for (int d = 0; d < ND; ++d) o[d] = f32x16{};
      m = -INFINITY;
      nmu = 0.f;
      l = 0.f;
      const int64_t first = kbeg + grp * BN;
      ks = Stream{reinterpret_cast<uint64_t>(kg + first * ks1), kr.keys - grp * BN, kbuf0};
      vs = Stream{reinterpret_cast<uint64_t>(vg + first * vs1), kr.keys - grp * BN, vbuf0};
      if (nkt > 0) {
        issue_k();
        issue_v();
        issue_k();
      }
      // The Q loads have landed before the walk (their first use inside it would put
      // their wait, and so a wait for the tile loads after them, into every iteration).
#pragma unroll
      for (int s = 0; s < NS; ++s) asm volatile("" : "+v"(qr[s]));
      f32x16 st[2][2];           // S^T of two consecutive tiles: [parity][32-key half]
      uint32_t kb = kl, vb = 0;  // this lane's K base of the next S tile, V offset of this tile

      // Tile t: K(t + 1) and V(t) have landed (every load so far), K(t + 2) goes into
      // the buffer of K(t), read an iteration ago, and V(t + 1) into that of V(t - 1).
      auto body = [&](auto par_tag, int t) __attribute__((always_inline)) {
        constexpr int PAR = decltype(par_tag)::value;
        constexpr DuoSeq<E> SEQ{};
        constexpr int LA = 3;  // operand reads run LA slots ahead of their MFMAs (2, 4 and 6: the same time)
        loads_done_barrier();
        issue_v();
        issue_k();
        mask(st[PAR], t);
        if (safe) {
          const float mx = row_max(st[PAR]);
          if (__any(mx > m + 8.f)) {
            const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - (mn == -INFINITY ? 0.f : mn));
            l *= alpha;
#pragma unroll
            for (int d = 0; d < ND; ++d) o[d] *= alpha;
            m = mn;
            nmu = mn == -INFINITY ? 0.f : -mn;
          }
        }
        bf16x8 op[SEQ.n];
        auto read = [&](int i) __attribute__((always_inline)) {
          if (SEQ.what[i] >= 0) op[i] = SEQ.what[i] < NS2 ? kread(kb, SEQ.what[i]) : vread(vb, SEQ.what[i] - NS2);
        };
#pragma unroll
        for (int i = 0; i < LA; ++i) read(i);
        __builtin_amdgcn_sched_barrier(0);
        // A slot: one MFMA, and the stages of the scores begun in it (exponent), one
        // slot before (exp2) and two slots before (row sum of the unrounded p, bf16).
        float sv[32], ev[32], ls = 0.f;
        uint32_t pw[16];
#pragma unroll
        for (int i = 0; i < SEQ.n; ++i) {
          if (i + LA < SEQ.n) read(i + LA);
#pragma unroll
          for (int x = 0; x < 32; ++x)
            if (SEQ.sl(x) == i - 2) {
              ls += ev[x];
              if (x & 1) pw[x >> 1] = pack_bf16x2(ev[x - 1], ev[x]);
            }
#pragma unroll
          for (int x = 0; x < 32; ++x)
            if (SEQ.sl(x) == i) sv[x] = fmaf(st[PAR][x >> 4][x & 15], p.c, nmu);
#pragma unroll
          for (int x = 0; x < 32; ++x)
            if (SEQ.sl(x) == i - 1) ev[x] = __builtin_amdgcn_exp2f(sv[x]);
          const int w = SEQ.what[i], q = w - NS2;
          if (w >= NS2)
            o[q % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                op[i], __builtin_bit_cast(bf16x8, u32x4{pw[4 * (q / ND)], pw[4 * (q / ND) + 1], pw[4 * (q / ND) + 2], pw[4 * (q / ND) + 3]}),
                o[q % ND], 0, 0, 0);
          else if (w >= 0)
            st[PAR ^ 1][w & 1] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(op[i], qr[w >> 1], w < 2 ? f32x16{} : st[PAR ^ 1][w & 1], 0, 0, 0);
          asm volatile("" : "+v"(ls));  // keeps the row sum's adds in their slots
          __builtin_amdgcn_sched_barrier(0);
        }
        l += ls;
        fine &= ls <= kHeadSum;
        kb = kb == kl ? kl + TB : kl;
        vb ^= TB;
      };

      int t = 0;
      if (nkt > 0) {
        loads_landed_barrier<2 * NL>();  // K(0) has landed
        auto first = [&]() __attribute__((always_inline)) {
#pragma unroll
          for (int q = 0; q < NS2; ++q)
            st[0][q & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kread(kb, q), qr[q >> 1], q < 2 ? f32x16{} : st[0][q & 1], 0, 0, 0);
          kb += TB;
          mask(st[0], 0);
          m = row_max(st[0]) + (safe ? 0.f : kMaxLift);
        };
        if (KG == 2) {
          if (nkt_w > 0) first();
          if (!safe) {  // group 0's max for both (a wave without a tile there has none here)
            float* fixed = reinterpret_cast<float*>(duo_smem + C::TILES) + 32 * wv + li;
            if (grp == 0) *fixed = m;
            __syncthreads();
            m = *fixed;
          }
        }
        if (nkt_w > 0) {
          if (KG == 1) first();
          nmu = m == -INFINITY ? 0.f : -m;
          // No finite logit among the first tile's visible keys: the max would be fixed
          // at 0, and p of later logits far below 0 flush.
          if (!safe) fine = m != -INFINITY || (p.causal && kbeg > r0 + li + diag);
          for (; t + 1 < nkt_w; t += 2) {
            body(std::integral_constant<int, 0>{}, t);
            body(std::integral_constant<int, 1>{}, t + 1);
          }
          if (t < nkt_w) {
            body(std::integral_constant<int, 0>{}, t);
            ++t;
          }
        }
      }
      for (; t < nkt; ++t) {  // tiles past this wave's rows: loads and barriers only
        loads_done_barrier();
        issue_v();
        issue_k();
      }
      __builtin_amdgcn_s_waitcnt(0x0f70);  // every direct load has landed
      return fine;
    };

    // One loop body serves both walks; the block takes the second where a wave failed.
    bool safe = false;
#pragma unroll 1
    for (;;) {
      const bool fine = walk(safe);
      __syncthreads();  // the tile buffers are free
      if (safe) break;
      uint32_t* failed = reinterpret_cast<uint32_t*>(duo_smem);
      const bool mine = __any(!fine);
      if (lane == 0) failed[wid] = mine;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < 4 * KG; ++w) safe |= failed[w] != 0;
      __syncthreads();
      if (!safe) break;
    }

    char* stage = duo_smem + wv * (KG == 2 ? C::MERGE : 32 * C::STAGE_ROW);
    if constexpr (KG == 2) {
      // Group 1's sums go through LDS to group 0, which merges and stores.
      float* mb = reinterpret_cast<float*>(stage) + lane;
      if (grp == 1) {
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) mb[64 * (16 * d + r)] = o[d][r];
        mb[64 * 16 * ND] = m;
        mb[64 * 16 * ND + 64] = l;
      }
      __syncthreads();
      if (grp == 1) continue;
      const float m1 = mb[64 * 16 * ND], mn = fmaxf(m, m1), mu = mn == -INFINITY ? 0.f : mn;
      const float w0 = __builtin_amdgcn_exp2f(m - mu), w1 = __builtin_amdgcn_exp2f(m1 - mu);
      l = l * w0 + mb[64 * 16 * ND + 64] * w1;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = o[d][r] * w0 + mb[64 * (16 * d + r)] * w1;
    }
    float lt = l + __shfl_xor(l, 32);
    if constexpr (SPLIT) {
      // The rows' partials for the combine: O unnormalised, m (scaled log2 units), l.
      const float f = level_partial(m, lt);
      const int row = r0 + li;
      if (row < L) {
        const int64_t slot = (((int64_t)dw.b * p.heads + dw.h) * p.seq_q + row) * gridDim.y + blockIdx.y;
        float* po = p.part_acc + slot * E + 4 * hf;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(po + 32 * d + 8 * q) = f32x4{o[d][4 * q] * f, o[d][4 * q + 1] * f, o[d][4 * q + 2] * f, o[d][4 * q + 3] * f};
        if (hf == 0) {
          p.part_ml[2 * slot] = m;
          p.part_ml[2 * slot + 1] = lt;
        }
      }
      continue;
    }
    // out = O / l, staged through this wave's part of the tile buffers so that each
    // store instruction writes whole rows (as store_staged).
    constexpr int CPR = C::CPR, RPI = 64 / CPR;
    const int ch = lane % CPR, rr0 = lane / CPR;
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    char* rowp = stage + li * C::STAGE_ROW;
    wave_lds_sync();  // the merge's reads before the staging overwrites them
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        u32x2 v = {pack_bf16x2(o[d][4 * q] * inv, o[d][4 * q + 1] * inv),
                   pack_bf16x2(o[d][4 * q + 2] * inv, o[d][4 * q + 3] * inv)};
        *reinterpret_cast<u32x2*>(rowp + (32 * d + 8 * q + 4 * hf) * 2) = v;
      }
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 32 / RPI; ++k) {
      const int rr = rr0 + RPI * k, row = r0 + rr;
      const u32x4 v = *reinterpret_cast<const u32x4*>(stage + rr * C::STAGE_ROW + ch * 16);
      if (row < L) __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(out + (int64_t)row * p.heads * E + ch * 8));
    }
  }
}

template <int E>
static int duo_launch(const FlashParams& p, const DuoPlan& d, hipStream_t stream) {
  using C1 = DuoCfg<E, 1>;
  using C2 = DuoCfg<E, 2>;
  if (d.splits > 1)
    return launch_lds(flash_duo_kernel<E, 1, true>, d.gx, 256, C1::LDS_BYTES, p, stream, d.splits, 0);
  if (d.kg == 2) return launch_lds(flash_duo_kernel<E, 2, false>, d.gx, 512, C2::LDS_BYTES, p, stream, 1, (int)d.pair);
  return launch_lds(flash_duo_kernel<E, 1, false>, d.gx, 256, C1::LDS_BYTES, p, stream, 1, (int)d.pair);
}

}  // namespace ca
