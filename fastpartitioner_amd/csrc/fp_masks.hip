// fp_masks.hip -- allocation and construction of the nets' part masks
// (fp_masks.h).
#include "fp_masks.h"

namespace fpe {
namespace {

constexpr int MASK_BLOCK = 256;
constexpr int MASK_SMALL = 8;  // lists of at most this many entries are taken by one lane each

// Each wave takes 64 consecutive nets, one per lane: a short list is turned
// into its record by its lane, the others by the wave in turn, through P-word
// bitmaps in LDS. The record past the last net is zeros. Bound by the reads of
// the lists and the writes of the records (16 P bytes per net).
__global__ void __launch_bounds__(MASK_BLOCK) k_build_masks(const unsigned* __restrict__ net_ptr,
                                                            const unsigned* __restrict__ ent, int noe, int P, int pb,
                                                            unsigned pmask, unsigned long long* __restrict__ masks) {
  __shared__ unsigned s_bits[MASK_BLOCK / WAVE][4 * MASK_PMAX];
  __shared__ unsigned s_lane[MASK_BLOCK][2 * MASK_PMAX + 1];  // odd: the lanes fall on distinct banks
  const int lane = lane_id(), nw = (int)(blockDim.x / WAVE);
  unsigned* bits = s_bits[wave_id()];
  if (blockIdx.x == 0 && (int)threadIdx.x < 2 * P) masks[(size_t)noe * (size_t)(2 * P) + threadIdx.x] = 0ull;
  for (int n0 = ((int)blockIdx.x * nw + wave_id()) * WAVE; n0 < noe; n0 += (int)gridDim.x * nw * WAVE) {
    const int n = n0 + lane;
    unsigned seg = 0;
    int L = 0;
    if (n < noe) {
      seg = net_ptr[n] + (unsigned)n;
      L = (int)ent[seg];
    }
    const bool mine = n < noe && L <= MASK_SMALL;
    unsigned x[MASK_SMALL];
#pragma unroll
    for (int t = 0; t < MASK_SMALL; t++) x[t] = mine && t < L ? ent[seg + 1 + (unsigned)t] : 0u;
    if (mine) lane_store_masks(x, L, pb, pmask, P, s_lane[threadIdx.x], masks + (size_t)n * (size_t)(2 * P));
    unsigned long long big = __ballot(n < noe && !mine);
    while (big) {
      const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)big) - 1);
      big &= big - 1;
      const unsigned sj = (unsigned)__builtin_amdgcn_readlane((int)seg, l);
      const int Lj = __builtin_amdgcn_readlane(L, l);
      if (lane < 4 * P) bits[lane] = 0u;
      wave_lds_sync();
      for (int t = lane; t < Lj; t += WAVE) {
        const unsigned y = ent[sj + 1 + (unsigned)t];
        const unsigned q = y & pmask, b = 1u << (q & 31u);
        atomicOr(&bits[q >> 5], b);
        if ((y >> pb) == 1u) atomicOr(&bits[2 * P + (int)(q >> 5)], b);
      }
      wave_lds_sync();
      unsigned* out = reinterpret_cast<unsigned*>(masks + (size_t)(n0 + l) * (size_t)(2 * P));
      if (lane < 4 * P) out[lane] = bits[lane];
      wave_lds_sync();
    }
  }
}

}  // namespace

unsigned long long* ensure_masks(fp_ctx* ctx) {
  const int P = mask_words(ctx->K);
  if (P == 0 || !ctx->use_masks) return nullptr;
  const size_t need = ((size_t)ctx->noe + 1) * (size_t)(2 * P);
  // the evaluation reads records and net ids at 32-bit byte offsets
  if (need * sizeof(unsigned long long) >= (size_t{1} << 32) || ctx->pins >= (1ll << 30)) return nullptr;
  if (need > ctx->mask_cap) {
    // a refinement rebuilds them: those of a smaller K are given back
    ctx->mask_cap = 0;
    if ((ctx->masks ? dgrow(ctx, &ctx->masks, need) : dalloc(ctx, &ctx->masks, need)) != FP_OK) return nullptr;
    ctx->mask_cap = need;
  }
  return ctx->masks;
}

void drop_masks(fp_ctx* ctx) {
  if (ctx->masks && dfree_own(ctx, ctx->masks)) {
    ctx->masks = nullptr;
    ctx->mask_cap = 0;
  }
}

void build_masks(fp_ctx* ctx, unsigned long long* masks) {
  const int grid = std::max(1, std::min((ctx->noe + MASK_BLOCK - 1) / MASK_BLOCK, 8192));
  k_build_masks<<<grid, MASK_BLOCK, 0, ctx->stream>>>(ctx->net_ptr, ctx->ent, ctx->noe, mask_words(ctx->K), ctx->pb,
                                                      ctx->pmask, masks);
}

}  // namespace fpe
