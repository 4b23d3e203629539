// fp_short.h -- evaluation of a vertex whose lists are few and short together,
// for K past the part masks' range.
//
// With K parts and few entries per net, a count per part and a scan of all K
// of them is mostly work for parts that no net lists: 16 steps of 64 parts at
// K = 1024 for the 150 entries of a vertex of 12 nets, and a 64-lane window for
// every list of a dozen entries. Here the lists are cut into rows of 16 words,
// four rows share a window, and the candidates are the entries themselves: a
// lane scores the part of its own entry from that part's count.
#pragma once
#include "fp_internal.h"

namespace fpe {

constexpr int SHORT_GROUP = 4;                // windows loaded together
constexpr int SHORT_WINDOWS = 2 * SHORT_GROUP;
constexpr int SHORT_ROWS = 4 * SHORT_WINDOWS;  // rows of a vertex at most

#ifdef __HIPCC__
// A row: its first word's offset, and net | place in the net's list << 6 |
// the list's length << 12. A list of L entries is (its length word included)
// ceil((L + 1) / 16) rows, none for L = 0.
struct ShortLists {
  unsigned x[SHORT_WINDOWS];  // lane 16 g + t of window i: word t of row 4 i + g
  unsigned in;                // bit i: the lane holds an entry of window i
  int nwin;
};

// The lists of deg nets, lane j holding net j's segment offset and length (0
// past deg). Returns false if they have more than SHORT_ROWS rows or the vertex
// more than 64 nets. rows (SHORT_ROWS words in LDS, the wave's own) keeps the
// rows for short_net. pad is the offset of the zero padding.
__device__ __forceinline__ bool short_load(const unsigned short* __restrict__ ev, unsigned sg, unsigned L, int deg,
                                           unsigned pad, uint2* rows, ShortLists& s) {
  const int lane = lane_id(), t = lane & 15;
  if (deg > WAVE) return false;
  const int nr = L ? (int)((L + 16u) >> 4) : 0;
  const int incl = wave_incl_scan(nr);
  const int total = __builtin_amdgcn_readlane(incl, WAVE - 1);
  if (total > SHORT_ROWS) return false;
  s.nwin = (total + 3) / 4;
  s.in = 0;
  if (lane >= total && lane < SHORT_ROWS) rows[lane] = make_uint2(pad, 0u);
  for (int c = 0; __ballot(c < nr); c++)
    if (c < nr) rows[incl - nr + c] = make_uint2(sg + 16u * (unsigned)c, (unsigned)(lane | (c << 6)) | (L << 12));
  wave_lds_sync();
  auto group = [&](int i0) {
    unsigned info[SHORT_GROUP];
#pragma unroll
    for (int i = 0; i < SHORT_GROUP; i++) {
      const uint2 r = rows[4 * (i0 + i) + (lane >> 4)];
      info[i] = r.y;
      s.x[i0 + i] = ev[r.x + (unsigned)t];
    }
#pragma unroll
    for (int i = 0; i < SHORT_GROUP; i++) {
      const unsigned at = ((info[i] >> 6) & 63u) * 16u + (unsigned)t;  // word of the net's segment
      s.in |= at >= 1u && at <= (info[i] >> 12) ? 1u << (i0 + i) : 0u;
    }
  };
  group(0);
  if (s.nwin > SHORT_GROUP) {
    group(SHORT_GROUP);
  } else {
#pragma unroll
    for (int i = SHORT_GROUP; i < SHORT_WINDOWS; i++) s.x[i] = 0;
  }
  return true;
}

// the net of this lane's entry of window i
__device__ __forceinline__ int short_net(const uint2* rows, int i) { return (int)(rows[4 * i + (lane_id() >> 4)].y & 63u); }

// f(window, word) for every window, the lanes without an entry masked off
template <class F>
__device__ __forceinline__ void short_each(const ShortLists& s, F f) {
#pragma unroll
  for (int i = 0; i < SHORT_GROUP; i++)
    if ((s.in >> i) & 1u) f(i, s.x[i]);
  if (s.nwin <= SHORT_GROUP) return;
#pragma unroll
  for (int i = SHORT_GROUP; i < SHORT_WINDOWS; i++)
    if ((s.in >> i) & 1u) f(i, s.x[i]);
}

// The LDG choice (mask_ldg's, fp_masks.h) among the parts the lists hold: the
// lexicographic max of (score, -size, -first rank) over score > 0, score =
// (count, less 1 for own) * penalty. An entry's rank is its row and its place
// there, the order in which the reference's scan meets the parts
// (TV/partition.cpp:318-338). cnt (K counts in LDS, the wave's own) is zero
// before and after. Returns the part and its count, or -1.
__device__ __forceinline__ int short_ldg(const ShortLists& s, unsigned* cnt, const double* s_pen,
                                         const unsigned* s_skey, int own, unsigned& craw) {
  const int lane = lane_id();
  short_each(s, [&](int, unsigned x) { atomicAdd(&cnt[x & ~EV_SINGLE], 1u); });
  wave_lds_sync();
  double best = 0;
  unsigned bkey = 0, bc = 0;
  int bq = -1, bi = 0;
  short_each(s, [&](int i, unsigned x) {
    const unsigned q = x & ~EV_SINGLE;
    const unsigned c = cnt[q], key = s_skey[q];
    const double sc = (double)((int)c - ((int)q == own ? 1 : 0)) * s_pen[q];
    // of one lane's entries of equal score and size the first keeps its place: it ranks first
    if (sc > best || (sc == best && key < bkey)) {
      best = sc;
      bkey = key;
      bq = (int)q;
      bc = c;
      bi = i;
    }
  });
  wave_lds_sync();
  short_each(s, [&](int, unsigned x) { cnt[x & ~EV_SINGLE] = 0u; });
  wave_lds_sync();
  const unsigned long long bb = (unsigned long long)__double_as_longlong(best);
  if (__ballot(bb != 0ull) == 0ull) return -1;
  unsigned long long cand = __ballot(bb == wave_max_u64(bb));
  int l = __ffsll((long long)cand) - 1;
  const int first = __builtin_amdgcn_readlane(bq, l);
  if (cand & __ballot(bq != first)) {
    // several parts share the best score: the lightest, then the first met
    const unsigned mk = wave_min_u32((cand >> lane) & 1ull ? bkey : ~0u);
    cand &= __ballot(bkey == mk);
    const unsigned rank = (unsigned)((4 * bi + (lane >> 4)) * 16 + (lane & 15));
    const unsigned mr = wave_min_u32((cand >> lane) & 1ull ? rank : ~0u);
    l = __ffsll((long long)(cand & __ballot(rank == mr))) - 1;
  }
  craw = (unsigned)__builtin_amdgcn_readlane((int)bc, l);
  return __builtin_amdgcn_readlane(bq, l);
}
#endif

}  // namespace fpe
