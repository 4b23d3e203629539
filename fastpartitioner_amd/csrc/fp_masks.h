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

constexpr int MASK_PMAX = 8;  // counts, penalties and size keys of 8 parts per lane fit 64 VGPRs
constexpr int MASK_KMAX = 64 * MASK_PMAX;

inline int mask_words(int K) { return K <= MASK_KMAX ? (K + 63) / 64 : 0; }

// The context's mask array for its K, or nullptr when K is above MASK_KMAX or
// the array cannot be allocated (the list evaluation then runs).
unsigned long long* ensure_masks(fp_ctx* ctx);
// Every record from the resident lists, on the context's stream.
void build_masks(fp_ctx* ctx, unsigned long long* masks);

#ifdef __HIPCC__
// c += this lane's bit of m (m wave-uniform): the bit is the add's carry-in
__device__ __forceinline__ void add_lane_bit(unsigned& c, unsigned long long m) {
  asm("v_addc_co_u32_e64 %0, vcc, 0, %0, %1" : "+v"(c) : "s"(m) : "vcc");
}
// c - this lane's bit of m
__device__ __forceinline__ unsigned sub_lane_bit(unsigned c, unsigned long long m) {
  unsigned r;
  asm("v_subbrev_co_u32_e64 %0, vcc, 0, %1, %2" : "=v"(r) : "v"(c), "s"(m) : "vcc");
  return r;
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
