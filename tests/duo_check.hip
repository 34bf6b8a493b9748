// Host-side address check of flash_duo_kernel (test infrastructure; compiled for the
// host and run by tests/test_duo_geometry.py), beside geom_check.hip: for every call
// shape on stdin that duo_plan takes, it replays duo_work, duo_keys, the tile windows
// and duo_tile_offset of every block, split, pass, key group, wave, tile and lane.
// Every query row is computed once per split, every wave walks exactly the tiles that
// hold a key one of its rows sees, the key groups cover them, every load lies in its
// tensor, and the swizzled LDS layout is a permutation of the tile whose operand reads
// hit the chunks that the loads filled.
//
// Input lines and --plant as geom_check.hip.  Output: "ok <taken> <accesses>".
// --plans: instead, per line "<key groups, 0: the 64-row kernel> <splits> <pairs>".
#include <stdio.h>
#include <string.h>

#include "../cpu-attention_amd/csrc/ca_flash.hip"
#include "../cpu-attention_amd/csrc/ca_rows.hip"
#include "../cpu-attention_amd/csrc/ca_small.hip"

#include <vector>

using namespace ca;

static long long g_checks = 0;
static bool g_plant = false;
static char g_fail[256];
#define FAIL(...)                                                    \
  do {                                                               \
    if (!g_fail[0]) snprintf(g_fail, sizeof g_fail, __VA_ARGS__);    \
    return false;                                                    \
  } while (0)

// The loads of the tile at key k0 of a stream whose range ends at kend.
template <int E, bool V>
static bool tile(int S, int64_t stride, int k0, int kend) {
  int bytes = tile_window<E>(kend - k0, 2 * (int)stride);
  if (g_plant && kend > k0 && kend - k0 < 64) bytes += 2 * (int)stride;
  for (int wv = 0; wv < 4; ++wv)
    for (int lane = 0; lane < 64; ++lane)
      for (int i = 0; i < DuoCfg<E, 1>::NL; ++i) {
        const uint32_t o = (uint32_t)duo_tile_offset<E, V>(wv, lane, i, (int)stride);
        if ((uint64_t)o + 16 > (uint64_t)bytes) continue;
        ++g_checks;
        const int64_t r = stride ? o / (2 * stride) : 0, within = o - r * 2 * stride;
        if (k0 < 0 || k0 + r >= S || within + 16 > 2 * E) FAIL("key %lld of %d", (long long)(k0 + r), S);
        if (k0 + r >= kend) FAIL("a load past the range's end outside the tensor's rows it may read");
      }
  return true;
}

// The LDS layout: chunk P of a tile holds (row, column chunk) duo_tile_offset names;
// the K and V^T operand addresses of the kernel must find theirs there.
template <int E>
static bool layout() {
  constexpr int CPR = E / 8, NS = E / 16, ND = E / 32;
  std::vector<int> kat(64 * CPR, -1), vat(64 * CPR, -1);  // (row * CPR + column) -> LDS chunk
  for (int wv = 0; wv < 4; ++wv)
    for (int lane = 0; lane < 64; ++lane)
      for (int i = 0; i < DuoCfg<E, 1>::NL; ++i) {
        const int P = (4 * i + wv) * 64 + lane;
        kat[duo_tile_offset<E, false>(wv, lane, i, E) / 16] = P;
        vat[duo_tile_offset<E, true>(wv, lane, i, E) / 16] = P;
      }
  for (int c : kat) if (c < 0) FAIL("K layout is no permutation");
  for (int c : vat) if (c < 0) FAIL("V layout is no permutation");
  for (int lane = 0; lane < 64; ++lane) {
    const int li = lane & 31, hf = lane >> 5, j = lane & 15, dh = (lane >> 4) & 1;
    for (int q = 0; q < 2 * NS; ++q) {
      const int a = ((li * 2 * E + ((hf ^ duo_k_swz<E>(li)) << 4)) ^ ((q >> 1) << 5)) + (q & 1) * 64 * E;
      if (a != 16 * kat[(li + 32 * (q & 1)) * CPR + 2 * (q >> 1) + hf]) FAIL("K operand %d of lane %d", q, lane);
    }
    for (int d = 0; d < ND; ++d)
      for (int cc = 0; cc < 4; ++cc)
        for (int u = 0; u < 2; ++u) {
          const int row = 16 * cc + 8 * u + 4 * hf + (j >> 2), byte = 64 * d + 32 * dh + 8 * (j & 3);
          const int a = (4 * hf + (j >> 2)) * 2 * E + ((d ^ duo_v_swz<E>(j >> 2)) << 6) + dh * 32 + (j & 3) * 8 + (16 * cc + 8 * u) * 2 * E;
          if (a != 16 * vat[row * CPR + byte / 16] + byte % 16) FAIL("V operand %d %d of lane %d", cc, d, lane);
        }
  }
  return true;
}

template <int E>
static void print_plan(const FlashParams& p) {
  const FlashPlan plan = flash_plan(p, E, true);
  if (plan.kind != kPlanBf16) return (void)puts("other route");
  const DuoPlan d = duo_plan(p, E, plan);
  printf("%d %d %d\n", d.kg, (int)(d.kg ? d.splits : plan.splits), d.kg ? d.pair : plan.pair);
}

template <int E>
static bool check(const FlashParams& p, bool& taken) {
  const FlashPlan plan = flash_plan(p, E, true);
  if (plan.kind != kPlanBf16) return true;
  const DuoPlan d = duo_plan(p, E, plan);
  if (!d.kg) return true;
  taken = true;
  if (!layout<E>()) return false;
  const int L = (int)p.seq_q, S = (int)p.seq_k, BM = DuoCfg<E, 1>::BM;
  const int64_t rows = p.batch * p.heads * L;
  if (d.splits < 1 || d.splits > plan.splits || (d.splits > 1 && (d.kg != 1 || d.pair))) FAIL("plan");
  if (d.splits > 1 && rows * plan.splits * (E + 2) * 4 > plan.need) FAIL("partials outside the workspace");
  std::vector<int> seen(rows * d.splits, 0);
  for (int64_t bx = 0; bx < d.gx; ++bx) {
    const DuoWork w = duo_work(p, BM, d.pair, (uint32_t)bx, (uint32_t)d.gx);
    if (w.b >= p.batch || w.h >= p.heads || w.n < 1 || w.n > 2) FAIL("work of block %lld", (long long)bx);
    for (int sp = 0; sp < d.splits; ++sp)
      for (int pass = 0; pass < w.n; ++pass) {
        const int q0 = (int)(pass ? w.qb1 : w.qb0) * BM;
        if (q0 >= L) FAIL("query block %d", q0);
        for (int wv = 0; wv < 4; ++wv) {
          const int r0 = q0 + 32 * wv, last = (L < r0 + 32 ? L : r0 + 32) - 1;
          for (int r = r0; r <= last; ++r) ++seen[((int64_t)(w.b * p.heads + w.h) * L + r) * d.splits + sp];
          const int window = window_bytes(((int64_t)(L - 1 - r0) * (int)p.qs[1] + E) * 2);  // of Q
          for (int li = 0; li < 32; ++li)
            for (int c = 0; c < E / 8; ++c) {
              const int64_t o = ((int64_t)li * p.qs[1] + 8 * c) * 2;
              if (o + 16 <= window && r0 + li >= L && p.qs[1] >= E) FAIL("Q row %d", r0 + li);
            }
          for (int grp = 0; grp < d.kg; ++grp) {
            const DuoKeys k = duo_keys(p, q0, r0, d.splits > 1, sp, (int)d.splits, d.kg, grp);
            if (k.nkt_w > k.nkt || (k.nkt > 0 && (k.kbeg < 0 || k.kbeg % 64 || k.kbeg + k.keys > S))) FAIL("keys");
            // the tiles that hold a key of [kbeg, kbeg + keys) that the wave's last row sees
            int sees = k.kbeg + k.keys;
            if (p.causal && last + 1 + S - L < sees) sees = last + 1 + S - L;
            const int n = last < r0 || sees <= k.kbeg ? 0 : (sees - k.kbeg + 63) / 64;
            if (k.nkt_w < (n - grp + d.kg - 1) / d.kg) FAIL("wave %d walks %d of %d tiles", wv, k.nkt_w, n);
            // loads: K one tile further than V, all of them through the group's windows
            if (wv == 0 && (w.h == 0 || w.h + 1 == p.heads) && k.nkt > 0)
              for (int t = 0; t < k.nkt + 2; ++t)
                if (!tile<E, false>(S, p.ks[1], k.kbeg + (t * d.kg + grp) * 64, k.kbeg + k.keys) ||
                    !tile<E, true>(S, p.vs[1], k.kbeg + (t * d.kg + grp) * 64, k.kbeg + k.keys))
                  return false;
          }
        }
      }
  }
  for (int s : seen) if (s != 1) FAIL("a row is computed %d times", s);
  return true;
}

int main(int argc, char** argv) {
  g_plant = argc > 1 && !strcmp(argv[1], "--plant");
  const bool plans = argc > 1 && !strcmp(argv[1], "--plans");
  long long n = 0, E, bf, causal, batch, sq, sk, h, qs[3], ks[3], vs[3];
  while (scanf("%lld %lld %lld %lld %lld %lld %lld %lld %lld %lld %lld %lld %lld %lld %lld %lld", &E, &bf, &causal,
               &batch, &sq, &sk, &h, &qs[0], &qs[1], &qs[2], &ks[0], &ks[1], &ks[2], &vs[0], &vs[1], &vs[2]) == 16) {
    FlashParams p{};
    p.batch = batch; p.seq_q = sq; p.seq_k = sk; p.heads = h; p.causal = (int)causal;
    for (int i = 0; i < 3; ++i) { p.qs[i] = qs[i]; p.ks[i] = ks[i]; p.vs[i] = vs[i]; }
    bool taken = false;
    if (plans) {
      E == 32 ? print_plan<32>(p) : E == 64 ? print_plan<64>(p) : print_plan<128>(p);
      continue;
    }
    if (bf && !(E == 32 ? check<32>(p, taken) : E == 64 ? check<64>(p, taken) : check<128>(p, taken))) {
      printf("FAIL E=%lld causal=%lld N=%lld L=%lld S=%lld H=%lld: %s\n", E, causal, batch, sq, sk, h, g_fail);
      return 1;
    }
    n += taken;
  }
  if (!plans) printf("ok %lld %lld\n", n, g_checks);
}
