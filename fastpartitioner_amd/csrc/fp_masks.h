// fp_masks.h -- the nets' part masks: a second view of the connectivity lists
// for evaluations with K <= MASK_KMAX parts.
//
// Net n's record is 2 P 64-bit words, P = ceil(K / 64), at masks[n * 2 P]:
//   word u < P      bit b: the net lists part 64 u + b
//   word P + u      bit b: it does, with exactly one pin
// A record of zeros follows the last net's (index noe: a list of length 0).
// The masks are built from the lists when a refinement is planned and rewritten
// by the kernels that edit lists during its passes; nothing keeps them between
// calls.
//
// Why: an evaluation needs, per vertex, in how many of its nets each part is
// listed. From the lists that is one 64-lane window and one LDS atomic per 63
// entries, about 15 vector instructions each. With a record in scalar
// registers a net is one vector add per 64 parts, its lane's bit taken as the
// carry-in (add_lane_bit), and the counts stay in registers.
#pragma once
#include "fp_internal.h"

namespace fpe {

// Counts, penalties, size keys and numbers of P parts take 5 P registers a lane, and
// a record 2 P scalar registers: at P = 8 the evaluations use their whole budget
// (80 vector registers at 6 waves per SIMD, 72 at 7 for P <= 6; two of them spill
// 12 bytes) with two records in flight. Past that one of the two would have
// to give; no larger P was measured.
constexpr int MASK_PMAX = 8;
constexpr int MASK_KMAX = 64 * MASK_PMAX;

inline int mask_words(int K) { return K <= MASK_KMAX ? (K + 63) / 64 : 0; }

// The context's mask array for its K, or nullptr when K is above MASK_KMAX or
// the array cannot be allocated (the list evaluation then runs).
unsigned long long* ensure_masks(fp_ctx* ctx);
// Gives the array back, if it is an allocation of its own; the next
// ensure_masks makes another.
void drop_masks(fp_ctx* ctx);
inline long long held_mask_bytes(const fp_ctx* ctx) { return (long long)(ctx->mask_cap * sizeof(unsigned long long)); }
// Every record from the resident lists, on the context's stream.
void build_masks(fp_ctx* ctx, unsigned long long* masks);

// Shape of the evaluations through the masks: each wave takes up to per_wave
// slots (at most one per lane), as many waves as fit the GPU at 7 per SIMD (the
// instances for more than 384 parts hold 6), or as grid_cap > 0 blocks hold,
// sharing the slots evenly. Twice
// as many waves cost a TV round of 16,384 slots 9% (each sets itself up for
// one or two vertices) and gain one of 262,144 1%.
inline int mask_eval_share(int nslots, int grid_cap, int waves_per_block) {
  const int waves = grid_cap > 0 ? std::min(7168, grid_cap * waves_per_block) : 7168;
  return std::max(1, std::min(WAVE, (nslots + waves - 1) / waves));
}
inline int mask_eval_grid(int nslots, int grid_cap, int waves_per_block) {
  const int per_block = mask_eval_share(nslots, grid_cap, waves_per_block) * waves_per_block;
  return std::max(1, (nslots + per_block - 1) / per_block);
}
// nets past which a vertex's records of more than 4 words are counted another way (mask_count_wide)
constexpr int MASK_WIDE = 512;
inline bool mask_wide(const fp_ctx* ctx) { return mask_words(ctx->K) > 4 && ctx->max_vdeg > (unsigned)MASK_WIDE; }
// the last element of vtx_nets, which bounds its reads a vertex ahead
inline unsigned mask_last_pin(const fp_ctx* ctx) { return (unsigned)std::max(ctx->pins - 1, 0ll); }

#ifdef __HIPCC__
// A wave's slots s0, s0 + stride, ..., at most one per lane, and their number
// ns: a whole round of the grid's waves apart. Vertices of many nets often have
// neighbouring numbers, and a wave of neighbouring slots took several of them
// one after another while the others were done: 60,000 vertices, the first 8 in
// 15,000 nets each, two rounds of TV at K = 512 22.0 -> 2.9 ms, of MSV at
// K = 1024 22.6 -> 5.3 ms. The blocks of one die take neighbouring slots, so that
// its L2 brings a line of headers once. Without such vertices 20 passes of
// 1,000,000 slots in rounds of 262,144 take 13.82 ms so, 13.88 with the blocks in
// launch order, and 13.71 with a wave's slots neighbouring.
__device__ __forceinline__ void wave_slots(int nslots, int& s0, int& stride, int& ns) {
  const int nw = (int)(blockDim.x / WAVE);
  const unsigned nb = gridDim.x, xcd = blockIdx.x % XCDS;
  const int b = (int)(xcd * (nb / XCDS) + min(xcd, nb % XCDS) + blockIdx.x / XCDS);
  s0 = b * nw + wave_id();
  stride = (int)gridDim.x * nw;
  // each lane looks at its own slot: a round of 2,048 slots, one per wave, takes
  // 4.22 us so and 4.45 with the number from a division
  ns = __popcll(__ballot((long long)s0 + (long long)lane_id() * stride < nslots));
}

// c += this lane's bit of m: the bit is the add's carry-in. m has to come from
// scalar loads and scalar instructions: a mask that a vector instruction wrote
// (a comparison, a ballot) may be read as a carry only two wait states later, and
// the compiler, which keeps them for its own instructions, does not look into
// this one. (For such a mask it makes the same instruction from c + (a == b).)
__device__ __forceinline__ void add_lane_bit(unsigned& c, unsigned long long m) {
  asm("v_addc_co_u32_e64 %0, vcc, 0, %0, %1" : "+v"(c) : "s"(m) : "vcc");
}

// The counts start at MASK_BIAS: count_double turns a biased count, or one
// less, into the signed number's double by one full-rate addition (2^52 + x has
// x in the low word; the conversion instruction takes four times as long).
constexpr unsigned MASK_BIAS = 0x80000000u;

__device__ __forceinline__ double count_double(unsigned x) {
  return __longlong_as_double((long long)((0x43300000ull << 32) | x)) - (4503599627370496.0 + 2147483648.0);
}

// Records of nets in flight per wave: their words (2 P SGPRs each) have to fit
// the scalar registers.
template <int P>
constexpr int mask_nets_in_flight() {
  return P <= 2 ? 8 : (P <= 4 ? 4 : (P <= 6 ? 3 : 2));
}

// nets per chunk of a vertex's nets: no batch reaches past the wave's last lane
template <int P>
constexpr int mask_chunk() {
  return (WAVE / mask_nets_in_flight<P>()) * mask_nets_in_flight<P>();
}

// the present words of the record at byte offset off, into scalar registers
template <int P>
__device__ __forceinline__ void mask_load(const unsigned long long* masks, unsigned off, unsigned long long (&w)[P]) {
#pragma unroll
  for (int u = 0; u < P; u++) w[u] = uniform_load_at<unsigned long long>(masks, off, u);
}

// UNCUT: only a net of one part keeps its bit
template <int P, bool UNCUT>
__device__ __forceinline__ void mask_filter(unsigned long long (&w)[P]) {
  if (!UNCUT) return;
  int c = 0;
#pragma unroll
  for (int u = 0; u < P; u++) c += (int)__popcll(w[u]);
#pragma unroll
  for (int u = 0; u < P; u++) w[u] = c == 1 ? w[u] : 0ull;
}

// Adds nn <= mask_chunk nets to the counts of the lane's parts: lane j holds
// the byte offset of net j's record. A batch's loads are all issued before the
// first is waited for.
template <int P, bool UNCUT>
__device__ __forceinline__ void mask_count(const unsigned long long* masks, unsigned off, int nn, unsigned (&cnt)[P]) {
  constexpr int NB = mask_nets_in_flight<P>();
  auto batch = [&](int j0, int n) {
    unsigned long long w[NB][P];
#pragma unroll
    for (int j = 0; j < NB; j++)
      if (j < n) mask_load<P>(masks, (unsigned)__builtin_amdgcn_readlane((int)off, j0 + j), w[j]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NB; j++)
      if (j < n) {
        mask_filter<P, UNCUT>(w[j]);
#pragma unroll
        for (int u = 0; u < P; u++) add_lane_bit(cnt[u], w[j][u]);
      }
  };
  int j0 = 0;
  for (; j0 + NB <= nn; j0 += NB) batch(j0, NB);
  if (j0 < nn) batch(j0, nn - j0);
}

// Past MASK_WIDE nets, for K > 256: of records of 5 to 8 words two or three in
// flight are all that the scalar registers hold, and a vertex of thousands of
// nets is a chain of their latencies. Here a load of the wave brings a dword
// a lane, G records at once, MASK_WIDE_LOADS loads in flight; a lane counts the
// bits of its dword in bytes (bit 8 i + k in byte i of word k), which go through
// LDS (MASK_WIDE_WORDS words, the wave's own) to the lanes of their parts before
// they can overflow. each(off) runs per 64 nets, lane j holding the byte offset of
// net j's record (the zero record past the last net).
// 60,000 vertices, the first 8 in 15,000 nets each, two rounds of 60,000 at
// K = 512: TV 2.90 -> 1.21 ms, MSRV in rounds of 16,384 4.7 -> 1.32; with 512
// nets each 0.24 -> 0.17 and 0.48 -> 0.36. The kernels that hold both ways of
// counting are slower on ordinary vertices (200,000 Zipf vertices, K = 512, MSRV
// 4.22 -> 4.42 ms; their registers spill), so they are instances of their own
// for hypergraphs with such a vertex.
constexpr int MASK_WIDE_LOADS = 4;
constexpr int MASK_WIDE_WORDS = 8 * WAVE;

template <int P, class Each>
__device__ __forceinline__ void mask_count_wide(const char* masks, const char* vtx_nets, unsigned vb, int deg,
                                                unsigned zero, unsigned* lds, unsigned (&cnt)[P], Each each) {
  constexpr int D = 2 * P, G = WAVE / D, LOADS = (WAVE + G - 1) / G;  // dwords of a record; loads of 64 nets
  const int lane = lane_id(), g = lane / D, t = lane - g * D;
  unsigned bytes[8];
#pragma unroll
  for (int k = 0; k < 8; k++) bytes[k] = 0u;
  auto flush = [&]() {
#pragma unroll
    for (int k = 0; k < 8; k++) lds[8 * lane + k] = bytes[k];
    wave_lds_sync();
    const int bit = lane & 31;
#pragma unroll 1
    for (int h = 0; h < G; h++)
#pragma unroll
      for (int u = 0; u < P; u++)
        cnt[u] += (lds[8 * (h * D + 2 * u + (lane >> 5)) + (bit & 7)] >> (bit & 24)) & 255u;
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 8; k++) bytes[k] = 0u;
  };
  int counted = 0;  // dwords a lane's bytes hold
  for (int c0 = 0; c0 < deg; c0 += WAVE) {
    const unsigned id = *reinterpret_cast<const unsigned*>(vtx_nets + (vb + (unsigned)min(c0 + lane, deg - 1)) * 4u);
    const unsigned off = c0 + lane < deg ? id * (16u * P) : zero;
    for (int i0 = 0; i0 < LOADS; i0 += MASK_WIDE_LOADS) {
      unsigned x[MASK_WIDE_LOADS];
#pragma unroll
      for (int i = 0; i < MASK_WIDE_LOADS; i++) {
        const int j = (i0 + i) * G + g;
        const unsigned o = (unsigned)__shfl((int)off, j & (WAVE - 1));
        x[i] = *reinterpret_cast<const unsigned*>(masks + ((g < G && j < WAVE ? o : zero) + 4u * (unsigned)t));
      }
#pragma unroll
      for (int i = 0; i < MASK_WIDE_LOADS; i++)
#pragma unroll
        for (int k = 0; k < 8; k++) bytes[k] += (x[i] >> k) & 0x01010101u;
    }
    each(off);
    counted += (LOADS + MASK_WIDE_LOADS - 1) / MASK_WIDE_LOADS * MASK_WIDE_LOADS;
    if (counted > 255 - 2 * MASK_WIDE_LOADS - LOADS) {
      flush();
      counted = 0;
    }
  }
  flush();
}

// The LDG choice of a vertex (its nets vtx_nets[vb .. vb + deg)) from its
// counts: the lexicographic max of (score, -size, -first appearance) over
// score > 0, score = (count, less 1 for own) * penalty, which equals the
// reference's scan over the parts it meets (TV/partition.cpp:98-116, :345).
// pen holds the penalties, negative ones as 0 (which no more makes a candidate),
// own is -1 for a vertex without a part. Returns pid of the part (lane l's
// pid[u] for part 64 u + l) and its count, or -1 when no part scores above 0.
template <int P, bool UNCUT>
__device__ __forceinline__ int mask_ldg(const unsigned long long* masks, const unsigned* vtx_nets,
                                        const unsigned* vtx_seg, const unsigned short* ev, unsigned vb, int deg,
                                        int own, const unsigned (&cnt)[P], const double (&pen)[P],
                                        const unsigned (&skey)[P], const int (&pid)[P], unsigned& craw) {
  const int lane = lane_id();
  double sc[P];
  double best = 0;
  const int mine = own - lane;  // 64 u where own is this lane's part u
#pragma unroll
  for (int u = 0; u < P; u++) {
    // a part in none of the nets scores 0, or (own) no more, and is no candidate
    sc[u] = count_double(cnt[u] - (mine == u * WAVE ? 1u : 0u)) * pen[u];
    best = fmax(best, sc[u]);
  }
  // the wave's best: positive doubles order like their bit patterns, the
  // high words first and the low words only where several lanes share it
  const unsigned long long bb = (unsigned long long)__double_as_longlong(best);
  const unsigned hi = (unsigned)(bb >> 32);
  const unsigned mh = wave_max_u32(hi);
  if (mh == 0 && __ballot(bb != 0ull) == 0ull) return -1;
  const unsigned long long hl = __ballot(hi == mh);
  unsigned ml;
  if (__popcll(hl) == 1)
    ml = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)bb, __ffsll((long long)hl) - 1);
  else
    ml = wave_max_u32(hi == mh ? (unsigned)bb : 0u);
  const double m1 = __longlong_as_double((long long)(((unsigned long long)mh << 32) | ml));
  unsigned long long tie[P];
  int ntie = 0;
#pragma unroll
  for (int u = 0; u < P; u++) {
    tie[u] = __ballot(sc[u] == m1);
    ntie += (int)__popcll(tie[u]);
  }
  if (ntie > 1) {
    // equal scores: the lightest part
    unsigned k2 = ~0u;
#pragma unroll
    for (int u = 0; u < P; u++) k2 = min(k2, sc[u] == m1 ? skey[u] : ~0u);
    const unsigned m2 = wave_min_u32(k2);
    ntie = 0;
#pragma unroll
    for (int u = 0; u < P; u++) {
      tie[u] &= __ballot(skey[u] == m2);
      ntie += (int)__popcll(tie[u]);
    }
    if (ntie > 1) {
      // equal sizes too: the part the reference's scan meets first, i.e. of the
      // first net that lists one of them, the earliest in its list
      // (TV/partition.cpp:318-338)
      for (int t = 0; t < deg; t++) {
        unsigned long long w[P];
        mask_load<P>(masks, uniform_load(vtx_nets + (vb + (unsigned)t)) * (16u * P), w);
        mask_filter<P, UNCUT>(w);
        int c = 0;
#pragma unroll
        for (int u = 0; u < P; u++) {
          w[u] &= tie[u];
          c += (int)__popcll(w[u]);
        }
        if (c == 0) continue;
        if (c > 1) {
          const unsigned seg = uniform_load(vtx_seg + (vb + (unsigned)t));
          const int L = (int)ev[seg];
          for (int t0 = 0; t0 < L; t0 += WAVE) {
            const int e = t0 + lane;
            const int q = e < L ? (int)(ev[seg + 1u + (unsigned)e] & ~EV_SINGLE) : 0;
            unsigned long long x = 0;
#pragma unroll
            for (int u = 0; u < P; u++) x = (q >> 6) == u ? w[u] : x;
            const unsigned long long hit = __ballot(e < L && ((x >> (q & (WAVE - 1))) & 1ull));
            if (hit) {
              const int f = __builtin_amdgcn_readlane(q, __ffsll((long long)hit) - 1);
#pragma unroll
              for (int u = 0; u < P; u++) w[u] = (f >> 6) == u ? 1ull << (f & (WAVE - 1)) : 0ull;
              break;
            }
          }
        }
#pragma unroll
        for (int u = 0; u < P; u++) tie[u] = w[u];
        break;
      }
    }
  }
  // one bit is left: its part and count, from the lane that holds them
  unsigned long long any = 0;
  int px = 0;
  unsigned cx = 0;
#pragma unroll
  for (int u = 0; u < P; u++) {
    any |= tie[u];
    const bool t = __builtin_amdgcn_inverse_ballot_w64(tie[u]);
    px = t ? pid[u] : px;
    cx = t ? cnt[u] : cx;
  }
  const int l = __ffsll((long long)any) - 1;
  craw = (unsigned)__builtin_amdgcn_readlane((int)cx, l) - MASK_BIAS;
  return __builtin_amdgcn_readlane(px, l);
}

// The lowest-index part of minimum size (TV/partition.cpp:118-132), by the
// whole wavefront.
__device__ __forceinline__ int wave_lightest_part(const long long* __restrict__ sizes, int K) {
  long long bs = LLONG_MAX;
  int bi = INT_MAX;
  for (int q = lane_id(); q < K; q += WAVE) {
    const long long sz = sizes[q];
    if (sz < bs || bi == INT_MAX) { bs = sz; bi = q; }
  }
  for (int off = WAVE / 2; off > 0; off >>= 1) {
    const long long os = __shfl_xor(bs, off);
    const int oi = __shfl_xor(bi, off);
    if (os < bs || (os == bs && oi < bi)) { bs = os; bi = oi; }
  }
  return __builtin_amdgcn_readfirstlane(bi);
}

// One lane's record from a list of at most N entries x[0 .. L) in registers
// (packed (count << pb) | part), assembled in the lane's own 2 P LDS words.
template <int N>
__device__ __forceinline__ void lane_store_masks(const unsigned (&x)[N], int L, int pb, unsigned pmask, int P,
                                                 unsigned* my, unsigned long long* __restrict__ out) {
  for (int h = 0; h < 2; h++) {  // the present words, then the single ones
    for (int w = 0; w < 2 * P; w++) my[w] = 0u;
#pragma unroll
    for (int t = 0; t < N; t++) {
      const unsigned q = x[t] & pmask;
      if (t < L && (h == 0 || (x[t] >> pb) == 1u)) my[q >> 5] |= 1u << (q & 31u);
    }
    for (int u = 0; u < P; u++) out[h * P + u] = ((unsigned long long)my[2 * u + 1] << 32) | my[2 * u];
  }
}

// One wavefront's record from list entries held a lane each (part key, pin
// count cnt, where `in`), assembled in 4 P LDS words of the wave's own.
__device__ __forceinline__ void wave_store_entry_masks(bool in, unsigned key, unsigned cnt, int P, unsigned* words,
                                                       unsigned long long* __restrict__ out) {
  const int lane = lane_id();
  if (lane < 4 * P) words[lane] = 0u;
  wave_lds_sync();
  if (in) {
    const unsigned bit = 1u << (key & 31u);
    atomicOr(&words[key >> 5], bit);
    if (cnt == 1u) atomicOr(&words[2 * P + (int)(key >> 5)], bit);
  }
  wave_lds_sync();
  if (lane < 4 * P) reinterpret_cast<unsigned*>(out)[lane] = words[lane];
  wave_lds_sync();
}

// One wavefront's record from a list in LDS, assembled in 4 P LDS words of the
// wave's own.
__device__ __forceinline__ void wave_store_list_masks(const unsigned* list, int L, int pb, unsigned pmask, int P,
                                                      unsigned* words, unsigned long long* __restrict__ out) {
  const int lane = lane_id();
  if (lane < 4 * P) words[lane] = 0u;
  wave_lds_sync();
  for (int t = lane; t < L; t += WAVE) {
    const unsigned x = list[t];
    const unsigned q = x & pmask, bit = 1u << (q & 31u);
    atomicOr(&words[q >> 5], bit);
    if ((x >> pb) == 1u) atomicOr(&words[2 * P + (int)(q >> 5)], bit);
  }
  wave_lds_sync();
  if (lane < 4 * P) reinterpret_cast<unsigned*>(out)[lane] = words[lane];
  wave_lds_sync();
}

// One wavefront's record from a list in LDS with its part -> position index
// (wave_index_set): lane l looks up parts l, l + 64, ...
__device__ __forceinline__ void wave_store_masks(const unsigned* list, const unsigned short* at, int K, int pb, int P,
                                                 unsigned long long* __restrict__ out) {
  const int lane = lane_id();
  for (int u = 0; u < P; u++) {
    const int q = u * WAVE + lane;
    const unsigned j = q < K ? at[q] : LIST_NONE;
    const bool in = j != LIST_NONE;
    const unsigned x = in ? list[j] : 0u;
    const unsigned long long pm = __ballot(in), sm = __ballot(in && (x >> pb) == 1u);
    if (lane == 0) {
      out[u] = pm;
      out[P + u] = sm;
    }
  }
}
#endif

}  // namespace fpe
