// fp_tv.hip -- TV refinement on the device (TV/partition.cpp:307-440 decisions,
// TV/partition.cpp:669-896 round schedule).
//
// One pass = rounds of R consecutive ordering positions. A round is:
//   k_tv_eval_masks  (K <= 512) scores a vertex per wavefront from its nets'
//                part masks (fp_masks.h): counts per part in registers, the
//                LDG2 decision by a lexicographic wave reduction (parts that
//                share the best score and size are told apart by where the
//                reference's scan meets them), then the TV gain test
//   k_tv_eval    (larger K) the same from the lists' 16-bit evaluation view:
//                one 128-byte read per net brings its lambda and first 63
//                entries, 3 nets in flight; the further windows of long
//                lists follow as one task list over all of the vertex's long
//                nets, 2 windows in flight; pin counts per part in LDS
//                Both write the slots' decisions and (BAL) the candidate
//                weights per (part, 64-slot tile); REF candidates stamp
//                their nets with the round's tag
//   k_bal_scan   BAL: per part, whether its candidates exceed cap - size, and
//                then an exclusive scan of its row of tile weights
//   k_bal_admit  BAL: prefix admission per part in ordering order, commit of
//                part vector and sizes; the admitted stamp their nets
//   k_apply      replays the round's moves on the lists (and masks) of the
//                stamped nets in ordering order: a lane per net of at most 8
//                pins, a wavefront per larger one (plus, for REF, the commit of
//                the part vector and the source-part sizes in extra blocks).
//                A stamp is a plain store; a list of the touched nets took an
//                atomic per workgroup on one counter, about 12 ns each one
//                after another (a 16,384-slot evaluation: 56 -> 17 us without)
#include "fp_masks.h"

namespace fpe {
namespace {

constexpr int EVAL_BLOCK = 256;  // 4 wavefronts
constexpr int TILE = 64;         // slots per admission tile
#ifndef FP_NETS_IN_FLIGHT
#define FP_NETS_IN_FLIGHT 3
#endif
constexpr int NETS_IN_FLIGHT = FP_NETS_IN_FLIGHT;  // segment head windows loaded together per wave
// nets per chunk of a vertex's net list: a multiple of NETS_IN_FLIGHT, so that
// no group of a chunk reaches past the wave's last lane (lanes from nn on hold
// the zero padding: lists of length 0)
constexpr int CHUNK = (WAVE / NETS_IN_FLIGHT) * NETS_IN_FLIGHT;
#ifndef FP_LONG_TASKS
#define FP_LONG_TASKS 2
#endif
constexpr int LONG_TASKS = FP_LONG_TASKS;  // windows of long lists (any of the chunk's nets) loaded together
constexpr int SCAN_RUN = 16;     // consecutive tiles per thread in the BAL scan
constexpr int APPLY_BLOCK = 256;
constexpr int SMALL_NET = 8;     // nets of at most this many pins are replayed one per lane
constexpr int APPLY_NET_BLOCKS = 2048;  // all resident at 8 waves per SIMD (8,192 cost 8 to 18%)
constexpr int APPLY_NETS = 512;    // nets per block of the apply at most
constexpr int APPLY_LIST_NETS = 4;  // and at least, of a list
constexpr int APPLY_LIST_NOE = 1 << 18, APPLY_LIST_RATIO = 32;  // apply_by_list
constexpr unsigned HUGE_NET = 256;  // nets of at least this many pins are replayed first
constexpr int APPLY_GROUP = 4;     // 64-rank windows of a net whose loads the apply issues together
constexpr int APPLY_TOGETHER = 8;  // moves of a window tried together (wave_ilist_moves)

struct EvalArgs {
  const unsigned* vtx_ptr;
  const unsigned* vtx_nets;
  const unsigned* vtx_seg;
  const unsigned short* ev;
  unsigned pad_seg;  // the 64 zero words after the last segment: a list of length 0
  const int* part;
  const int* order;  // nullable: identity
  const int* vwgt;   // nullable: unit
  const long long* sizes;
  int K, pb;
  unsigned pmask;
  int r0, nslots, ntiles;
  double C;
  long long max_pw, min_pw;
  int* slot_own;
  int* slot_dec;
  int* dec_out;   // nullable (fp_eval_moves)
  int* gain_out;  // nullable
  // the round's tag goes to the stamps of the nets its candidates touch (nullable: no stamping)
  unsigned tag;
  unsigned* net_stamp;
  // BAL (nullable): candidate weight per (part, tile); frozen sizes copy
  int* hist;
  long long* sizes_frozen;
  // initial partition (nullable): the lowest-index part of minimum frozen size
  int* fb_out;
  // the nets' part masks (k_tv_eval_masks)
  const unsigned long long* masks;
  int noe;
  unsigned last_pin;  // the last element of vtx_nets
};

// slot decision of an unplaced vertex whose part the fallback assigns
constexpr int SLOT_FALLBACK = -2;

// The LDG2 decision of one vertex with first-appearance ranks, for a vertex
// whose best (score, size) two parts share: its lists are swept again into
// pin counts and ranks (i << pb | t, i the net's index in the vertex's list,
// t the part's position in the net's list: the order in which the reference's
// scan meets the parts, TV/partition.cpp:318-338), and the lexicographic max
// of (score, -size, -rank) over score > 0 picks the part. cnt and first are
// left clear (0, NOFIRST).
template <int MODE>
__device__ __forceinline__ void tie_decision(const EvalArgs& a, unsigned vb, int deg, int own, unsigned* cnt,
                                          unsigned* first, const double* s_pen, const unsigned* s_skey, int& d,
                                          unsigned& craw) {
  const int lane = lane_id(), K = a.K;
  for (int c0 = 0; c0 < deg; c0 += WAVE) {
    const int nn = min(WAVE, deg - c0);
    const unsigned sg = lane < nn ? a.vtx_seg[vb + (unsigned)(c0 + lane)] : a.pad_seg;
    wave_sweep_lists<1, 1>(a.ev, sg, nn, [&](int j, int L, int t, bool ok, unsigned x) {
      if (ok && (MODE != 2 || L == 1)) {  // mode 2, CN's stream: uncut nets only
        const int q = (int)(x & ~EV_SINGLE);
        atomicAdd(&cnt[q], 1u);
        atomicMin(&first[q], ((unsigned)(c0 + j) << a.pb) | (unsigned)t);
      }
    });
  }
  wave_lds_sync();
  unsigned long long b1 = 0, b2 = ~0ull;
  int bq = -1;
  unsigned bc = 0;
  for (int q = lane; q < K; q += WAVE) {
    const unsigned c = cnt[q], f = first[q];
    cnt[q] = 0;
    first[q] = NOFIRST;
    const int adj = (int)c - (q == own ? 1 : 0);
    const double sc = (double)adj * s_pen[q];
    const bool ok = c != 0 && sc > 0;
    const unsigned long long k1 = ok ? (unsigned long long)__double_as_longlong(sc) : 0ull;
    const unsigned long long k2 = ((unsigned long long)s_skey[q] << 32) | f;
    const bool better = ok && (k1 > b1 || (k1 == b1 && k2 < b2));
    b1 = better ? k1 : b1;
    b2 = better ? k2 : b2;
    bq = better ? q : bq;
    bc = better ? c : bc;
  }
  const unsigned long long m1 = wave_max_u64(b1);
  const unsigned long long m2 = wave_min_u64(b1 == m1 ? b2 : ~0ull);
  const int wl = __ffsll((long long)__ballot(b1 == m1 && b2 == m2)) - 1;
  d = __builtin_amdgcn_readlane(bq, wl);
  craw = (unsigned)__builtin_amdgcn_readlane((int)bc, wl);
  wave_lds_sync();
}

// The evaluation's modes: a refinement round (TV/partition.cpp:732-805), or a
// sub-round of the streaming initial partition, whose unplaced vertices
// (part -1) are scored over every list of their nets (LDG2,
// TV/partition.cpp:214-233; plain LDG, MGV/partition.cpp:28-65) or only over
// the lists of their uncut nets (CN/partition.cpp:138-156).
enum EvalMode { EVAL_REFINE = 0, EVAL_INIT = 1, EVAL_INIT_CN = 2 };

// Per vertex: sweep, LDG2 decision, TV gain test (TV/partition.cpp:732-805).
// Eight waves per SIMD (the hardware's maximum) hide more of the dependent
// list reads than the registers a freer allocation would save: the compiler
// keeps within 64 VGPRs by parking cold scalar values in VGPR lanes.
// EVAL_INIT*: a vertex already placed is skipped (no candidate); an unplaced
// one is a candidate for its LDG choice, the lowest-index part of minimum
// size standing in where the choice is above max_pw (where the reference
// would index part_sizes[-1]); the min_pw band does not apply (own == -1).
template <int MODE>
__global__ void __launch_bounds__(EVAL_BLOCK) __attribute__((amdgpu_waves_per_eu(8))) k_tv_eval(EvalArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int K = a.K;
  double* s_pen = reinterpret_cast<double*>(lds);
  unsigned* s_skey = reinterpret_cast<unsigned*>(s_pen + K);  // size_key of each frozen part size
  unsigned* wbase = s_skey + K;
  __shared__ long long red_sz[EVAL_BLOCK / WAVE];
  __shared__ int red_ix[EVAL_BLOCK / WAVE];
  const int lane = lane_id(), wave = wave_id(), nw = (int)(blockDim.x / WAVE);
  // per wavefront: cnt[K] and first[K], each followed by 64 spare slots that
  // take the atomics of lanes past a list's end (no branch around them)
  unsigned* cnt = wbase + (size_t)wave * 2 * (size_t)(K + WAVE);
  unsigned* first = cnt + K + WAVE;
  const int spare = K + lane_id();

  // penalties of the frozen part sizes: penalty = 1 - (1.0 * size / C)  (TV/partition.cpp:103)
  long long bs = LLONG_MAX;
  int bi = INT_MAX;
  for (int q = (int)threadIdx.x; q < K; q += (int)blockDim.x) {
    const long long sz = a.sizes[q];
    s_skey[q] = size_key(sz);
    s_pen[q] = 1.0 - ((double)sz / a.C);
    if (sz < bs) { bs = sz; bi = q; }
    if (blockIdx.x == 0 && a.sizes_frozen) a.sizes_frozen[q] = sz;
  }
  for (int q = lane; q < K; q += WAVE) { cnt[q] = 0; first[q] = NOFIRST; }
  // fallback: lowest-index part of minimum size (TV/partition.cpp:118-132)
  for (int off = WAVE / 2; off > 0; off >>= 1) {
    const long long os = __shfl_xor(bs, off);
    const int oi = __shfl_xor(bi, off);
    if (os < bs || (os == bs && oi < bi)) { bs = os; bi = oi; }
  }
  if (lane == 0) { red_sz[wave] = bs; red_ix[wave] = bi; }
  __syncthreads();
  int fb = red_ix[0];
  {
    long long b = red_sz[0];
    for (int w = 1; w < nw; w++)
      if (red_sz[w] < b || (red_sz[w] == b && red_ix[w] < fb)) { b = red_sz[w]; fb = red_ix[w]; }
  }
  if (MODE != EVAL_REFINE && blockIdx.x == 0 && threadIdx.x == 0) *a.fb_out = fb;

  // One wavefront per vertex, grid-stride over the round's slots, software
  // pipelined over the wave's vertices: while vertex X is swept, the segment
  // addresses of X+1's nets and the vertex header of X+2 are in flight.
  const int stride = (int)gridDim.x * nw;
  const int slot_end = a.nslots;
  int slot = (int)blockIdx.x * nw + wave;
  int hv[3], hown[3], hdeg[3];
  unsigned hvb[3];
  auto load_vertex = [&](int k, int sl) {
    if (sl < slot_end) {
      const int vv = a.order ? uniform_load(a.order + (a.r0 + sl)) : a.r0 + sl;
      hv[k] = vv;
      hown[k] = uniform_load(a.part + vv);
      hvb[k] = uniform_load(a.vtx_ptr + vv);
      hdeg[k] = (int)(uniform_load(a.vtx_ptr + vv + 1) - hvb[k]);
    } else {
      hv[k] = 0; hown[k] = 0; hvb[k] = 0; hdeg[k] = 0;
    }
  };
  auto load_segs = [&](int k) -> unsigned {
    return lane < min(hdeg[k], CHUNK) ? a.vtx_seg[hvb[k] + (unsigned)lane] : a.pad_seg;
  };
  // the first window group of the vertex about to be swept, loaded while the
  // previous vertex picks its candidate
  unsigned xpre[NETS_IN_FLIGHT];
  auto load_first = [&](unsigned sgv) {
#pragma unroll
    for (int u = 0; u < NETS_IN_FLIGHT; u++) {
      const unsigned sj = (unsigned)__builtin_amdgcn_readlane((int)sgv, u);
      xpre[u] = a.ev[sj + (unsigned)lane];
    }
  };
  load_vertex(0, slot);
  load_vertex(1, slot + stride);
  unsigned sg0 = load_segs(0);
  load_first(sg0);
  while (slot < slot_end) {
    load_vertex(2, slot + 2 * stride);
    const unsigned sg1 = load_segs(1);
    const int v = hv[0], own = hown[0], deg = hdeg[0];
    const unsigned vb = hvb[0];

    // sweep: histogram of parts over the lists of v's nets. The first
    // appearance of a part is ranked by (net index i in v's net list, position
    // t in that net's list), packed as i << pb | t (t < lambda <= K <= 2^pb):
    // the order in which the reference's scan meets the parts
    // (TV/partition.cpp:318-338). One 64-word read of a segment brings lambda
    // (lane 0) and the first 63 entries (lanes 1..63); NETS_IN_FLIGHT such
    // reads are issued together, longer lists are finished after. Lanes past
    // the vertex's nets hold the zero padding's offset, so the windows past
    // the last net see lambda = 0. The leave-gain count is kept per lane.
    int lgl = 0;
    for (int c0 = 0; c0 < deg; c0 += CHUNK) {
      const int nn = min(CHUNK, deg - c0);
      const unsigned sg = c0 == 0 ? sg0 : (lane < nn ? a.vtx_seg[vb + (unsigned)(c0 + lane)] : a.pad_seg);
      int lmax = 0;  // longest list of the chunk
      int lj = 0;    // lane j: lambda of the chunk's net j
      // the next group's windows are in flight while a group is counted
      unsigned xv[NETS_IN_FLIGHT];
      auto load_group = [&](int j0, unsigned (&dst)[NETS_IN_FLIGHT]) {
#pragma unroll
        for (int u = 0; u < NETS_IN_FLIGHT; u++) {
          const unsigned sj = (unsigned)__builtin_amdgcn_readlane((int)sg, j0 + u);
          dst[u] = a.ev[sj + (unsigned)lane];
        }
      };
      if (c0 == 0) {
#pragma unroll
        for (int u = 0; u < NETS_IN_FLIGHT; u++) xv[u] = xpre[u];
      } else {
        load_group(0, xv);
      }
      for (int j0 = 0; j0 < nn; j0 += NETS_IN_FLIGHT) {
        unsigned xn[NETS_IN_FLIGHT];
        const bool more = j0 + NETS_IN_FLIGHT < nn;
        if (more) load_group(j0 + NETS_IN_FLIGHT, xn);
#pragma unroll
        for (int u = 0; u < NETS_IN_FLIGHT; u++) {
          const int j = j0 + u;
          const int Lj = __builtin_amdgcn_readlane((int)xv[u], 0);
          lmax = max(lmax, Lj);
          lj = lane == j ? Lj : lj;
          const int t = lane - 1;
          // EVAL_INIT_CN: only nets of one part vote (lambda == 1)
          const bool ok = lane >= 1 && t < Lj && (MODE != EVAL_INIT_CN || Lj == 1);
          const unsigned x = xv[u];
          const int q = (int)(x & ~EV_SINGLE);
          const int qs = ok ? q : spare;
          atomicAdd(&cnt[qs], 1u);
          // leave gain: nets where v is the only pin of its part (TV/partition.cpp:365-368)
          lgl += ok && q == own && (x & EV_SINGLE) ? 1 : 0;
        }
        if (more) {
#pragma unroll
          for (int u = 0; u < NETS_IN_FLIGHT; u++) xv[u] = xn[u];
        }
      }
      // the rest of the long lists (more than 63 entries): entries 63.. in
      // windows of 64. Each (net, window) pair of the chunk is a task,
      // numbered net by net by a scan of the per-net window counts, and
      // LONG_TASKS tasks' windows are loaded together, whichever nets they
      // belong to; the lambdas come from the first windows.
      if (MODE != EVAL_INIT_CN && lmax > WAVE - 1) {
        const int nwin = lj >> 6;  // ceil((lambda - 63) / 64) windows past the first
        const int incl = wave_incl_scan(nwin);
        const int ntask = __builtin_amdgcn_readlane(incl, WAVE - 1);
        for (int k0 = 0; k0 < ntask; k0 += LONG_TASKS) {
          unsigned xw[LONG_TASKS];
          int tj[LONG_TASKS], tw[LONG_TASKS], tl[LONG_TASKS];
#pragma unroll
          for (int u = 0; u < LONG_TASKS; u++) {
            // past the last task: a repeat of it, with no entries counted
            const int k = min(k0 + u, ntask - 1);
            const int j = (int)__popcll(__ballot(incl <= k));  // its net: incl is non-decreasing
            const int w = k - __builtin_amdgcn_readlane(incl - nwin, j);
            const unsigned sj = (unsigned)__builtin_amdgcn_readlane((int)sg, j);
            const int Lj = __builtin_amdgcn_readlane(lj, j);
            tj[u] = j;
            tw[u] = WAVE - 1 + w * WAVE;
            tl[u] = k0 + u < ntask ? Lj : 0;
            const int t = tw[u] + lane;
            xw[u] = a.ev[sj + 1u + (unsigned)(t < Lj ? t : 0)];
          }
#pragma unroll
          for (int u = 0; u < LONG_TASKS; u++) {
            const int t = tw[u] + lane;
            const bool ok = t < tl[u];
            const unsigned x = xw[u];
            const int q = (int)(x & ~EV_SINGLE);
            const int qs = ok ? q : spare;
            atomicAdd(&cnt[qs], 1u);
            lgl += ok && q == own && (x & EV_SINGLE) ? 1 : 0;
          }
        }
      }
    }
    const int lg = wave_sum(lgl);
    load_first(sg1);
    wave_lds_sync();
    // candidates: lexicographic max of (score, -size, -first rank) over score >
    // 0 equals the sequential LDG2 scan over the active parts
    // (TV/partition.cpp:98-116). Scores are positive doubles, so their bit
    // patterns order like the values: key1 = score bits (max), key2 =
    // size_key(size) << 32 | first rank (min among key1 ties).
    const unsigned cfb = cnt[fb];
    // candidates: lexicographic max of (score, -size, -first rank) over score >
    // 0 (TV/partition.cpp:98-116). The first rank decides only between parts
    // of equal score and size: the sweep counts pins only, and a vertex whose
    // best (score, size) is shared by two parts is decided again with ranks
    // (tie_decision). Scores are positive doubles, so their bit patterns order
    // like the values: key1 = score bits (max), key2 = size_key(size) (min
    // among key1 ties); ltie: this lane met its best keys twice.
    unsigned long long b1 = 0;
    unsigned b2 = ~0u;
    int bq = -1;
    unsigned bc = 0;
    bool ltie = false;
    // four 64-part chunks per step, without branches: their LDS reads issue
    // together; every slot is cleared for the next vertex
    for (int q0 = 0; q0 < K; q0 += 4 * WAVE) {
      unsigned cv[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int q = min(q0 + u * WAVE + lane, K - 1);
        cv[u] = q0 + u * WAVE + lane < K ? cnt[q] : 0u;
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int q = q0 + u * WAVE + lane;
        const int qc = min(q, K - 1);
        if (q < K) cnt[q] = 0;
        const int adj = (int)cv[u] - (q == own ? 1 : 0);   // scores[part_id]-- (TV/partition.cpp:345)
        const double sc = (double)adj * s_pen[qc];
        const bool ok = cv[u] != 0 && sc > 0;
        const unsigned long long k1 = ok ? (unsigned long long)__double_as_longlong(sc) : 0ull;
        const unsigned k2 = s_skey[qc];
        const bool better = ok && (k1 > b1 || (k1 == b1 && k2 < b2));
        const bool same = ok && k1 == b1 && k2 == b2;
        ltie = better ? false : (ltie || same);
        b1 = better ? k1 : b1;
        b2 = better ? k2 : b2;
        bq = better ? q : bq;
        bc = better ? cv[u] : bc;
      }
    }
    const unsigned long long m1 = wave_max_u64(b1);
    wave_lds_sync();
    int d = fb;
    unsigned craw = cfb;
    if (m1 != 0) {
      // the second key is needed only when several lanes hold the best score
      unsigned long long cand = __ballot(b1 == m1);
      if (__popcll(cand) > 1) {
        const unsigned m2 = wave_min_u32(b1 == m1 ? b2 : ~0u);
        cand = __ballot(b1 == m1 && b2 == m2);
      }
      const int wl = __ffsll((long long)cand) - 1;
      if (__popcll(cand) > 1 || __builtin_amdgcn_readlane((int)ltie, wl)) {
        tie_decision<MODE>(a, vb, deg, own, cnt, first, s_pen, s_skey, d, craw);
      } else {
        d = __builtin_amdgcn_readlane(bq, wl);
        craw = (unsigned)__builtin_amdgcn_readlane((int)bc, wl);
      }
    }
    // the bands, compared as size keys (the same order)
    bool accept;
    int dd;  // the slot's decision: a part, -1 (none) or SLOT_FALLBACK
    if (MODE == EVAL_REFINE) {
      if (s_skey[d] > size_key(a.max_pw)) d = own;   // TV/partition.cpp:135-138
      if (s_skey[d] < size_key(a.min_pw)) d = own;   // TV/partition.cpp:140-143
      const int al = deg - (int)craw;      // arrival loss: nets of v lacking d (TV/partition.cpp:369-377)
      accept = d != own && lg >= al;       // TV/partition.cpp:380
      dd = accept ? d : -1;
    } else {
      // an unplaced vertex with no part above score 0, or whose choice is
      // above the band, takes its turn in the fallback
      accept = own < 0;
      dd = !accept ? -1 : (m1 == 0 || s_skey[d] > size_key(a.max_pw) ? SLOT_FALLBACK : d);
    }
    if (lane == 0) {
      a.slot_own[slot] = own;
      a.slot_dec[slot] = dd;
      if (MODE == EVAL_REFINE && a.dec_out) a.dec_out[v] = d;
      if (MODE == EVAL_REFINE && a.gain_out) a.gain_out[v] = d == own ? INT_MIN : lg - (deg - (int)craw);
      if (dd >= 0 && a.hist) {
        const int w = a.vwgt ? a.vwgt[v] : 1;
        atomicAdd(&a.hist[(size_t)d * (size_t)a.ntiles + (size_t)(slot / TILE)], w);
      }
    }
    if (accept && a.net_stamp) wave_stamp_nets(a.vtx_nets + vb, deg, a.tag, a.net_stamp);
    slot += stride;
    hv[0] = hv[1]; hown[0] = hown[1]; hvb[0] = hvb[1]; hdeg[0] = hdeg[1];
    hv[1] = hv[2]; hown[1] = hown[2]; hvb[1] = hvb[2]; hdeg[1] = hdeg[2];
    sg0 = sg1;
  }
}

// k_tv_eval through the nets' part masks (fp_masks.h), for K <= 64 P: lane l
// counts parts l, l + 64, ... of the vertex in registers. Per net a record's
// P present words come into scalar registers and are added with the lane's
// bit as the carry-in; the penalties and counts of a lane's parts stay in
// registers, so the sweep and the LDG scan touch no LDS. The single bit of the
// vertex's own part comes from one word per net, a net per lane.
// A wave takes slots a round of the grid's waves apart: their headers are loaded a slot per
// lane, their decisions written a slot per lane at the end. Both the vector
// and the scalar unit are near their issue limit here, so addresses are 32-bit
// offsets (the host checks the arrays' sizes) and everything per vertex that
// a lane can hold is held by one.
// The decision, the gain test and everything written are k_tv_eval's.
// WIDE: for hypergraphs with a vertex of more than MASK_WIDE nets (mask_count_wide).
template <int P, int MODE, bool WIDE>
__global__ void __launch_bounds__(EVAL_BLOCK) __attribute__((amdgpu_waves_per_eu(P <= 6 ? 7 : 6, P <= 6 ? 7 : 6))) k_tv_eval_masks(EvalArgs a) {
  constexpr int CH = mask_chunk<P>();
  constexpr unsigned ROW = 16u * P;  // bytes of a record
  static_assert(!WIDE || MODE != EVAL_INIT_CN, "uncut nets only: not a count of whole records");
  __shared__ double s_pen[64 * P];
  __shared__ unsigned s_skey[64 * P];
  __shared__ unsigned s_wide[WIDE ? EVAL_BLOCK / WAVE : 1][WIDE ? MASK_WIDE_WORDS : 1];
  const int K = a.K;
  const int lane = lane_id(), wave = wave_id();
  int s0, stride, ns;
  wave_slots(a.nslots, s0, stride, ns);
  const int slot_l = s0 + lane * stride;

  // lane i: the wave's slot i's vertex, its part and its net range
  int v_l = 0, own_l = 0;
  unsigned vb_l = 0, ve_l = 0;
  if (lane < ns) {
    const int z = a.r0 + slot_l;
    v_l = a.order ? a.order[z] : z;
    own_l = a.part[v_l];
    vb_l = a.vtx_ptr[v_l];
    ve_l = a.vtx_ptr[v_l + 1];
  }
  // penalties of the frozen part sizes: penalty = 1 - (1.0 * size / C)  (TV/partition.cpp:103)
  for (int q = (int)threadIdx.x; q < 64 * P; q += (int)blockDim.x) {
    const long long sz = q < K ? a.sizes[q] : 0;
    s_skey[q] = size_key(sz);
    s_pen[q] = q < K ? fmax(1.0 - ((double)sz / a.C), 0.0) : 0.0;
    if (blockIdx.x == 0 && a.sizes_frozen && q < K) a.sizes_frozen[q] = sz;
  }
  if (MODE != EVAL_REFINE && blockIdx.x == 0 && wave == 0) {
    const int fb = wave_lightest_part(a.sizes, K);
    if (lane == 0) *a.fb_out = fb;
  }
  __syncthreads();
  // per part of the lane: penalty, size key, and the part's number with bit 16
  // set where its size lies within the bands (compared as size keys, the same order)
  double pen[P];
  unsigned skey[P];
  int pid[P];
  auto load_parts = [&]() {
#pragma unroll
    for (int u = 0; u < P; u++) {
      pen[u] = s_pen[u * WAVE + lane];
      skey[u] = s_skey[u * WAVE + lane];
      const bool in = skey[u] <= size_key(a.max_pw) && (MODE != EVAL_REFINE || skey[u] >= size_key(a.min_pw));
      pid[u] = (u * WAVE + lane) | (in ? 1 << 16 : 0);
    }
  };
  load_parts();
  const char* masks = reinterpret_cast<const char*>(a.masks);
  // lane j: net j of slot i's vertex; past its last net some other net.
  // Loaded a vertex ahead, by every lane (a load that a branch may skip could
  // only be waited for together with the ones after it).
  const char* nets = reinterpret_cast<const char*>(a.vtx_nets);
  auto load_nets = [&](int i) -> unsigned {
    const unsigned k = (unsigned)__builtin_amdgcn_readlane((int)vb_l, i) + (unsigned)lane;
    return *reinterpret_cast<const unsigned*>(nets + min(k, a.last_pin) * 4u);
  };

  int dec_l = -1;  // lane i: slot i's decision: a part, -1 (none) or SLOT_FALLBACK
  // the headers have arrived before the loop (else its first wait would take in the loads of every turn)
  asm volatile("" ::"v"(own_l), "v"(vb_l), "v"(ve_l));
  unsigned id = ns > 0 ? load_nets(0) : 0u;
  for (int i = 0; i < ns; i++) {
    const unsigned id_next = load_nets(min(i + 1, ns - 1));
    const int own = __builtin_amdgcn_readlane(own_l, i);
    const unsigned vb = (unsigned)__builtin_amdgcn_readlane((int)vb_l, i);
    const int deg = (int)((unsigned)__builtin_amdgcn_readlane((int)ve_l, i) - vb);
    const unsigned id0 = id;
    id = id_next;
    if (MODE != EVAL_REFINE && own >= 0) continue;  // already placed

    unsigned cnt[P];
#pragma unroll
    for (int u = 0; u < P; u++) cnt[u] = MASK_BIAS;
    int lg = 0;  // leave gain: nets where v is the only pin of its part (TV/partition.cpp:365-368)
    // nn <= CH nets of the vertex, lane j's the one with id ids
    auto count_nets = [&](unsigned ids, int nn) {
      const unsigned off = (lane < nn ? ids : (unsigned)a.noe) * ROW;  // past the last net: the zero record
      unsigned sw = 0;
      if (MODE == EVAL_REFINE)
        sw = *reinterpret_cast<const unsigned*>(masks + (8u * P + 4u * (unsigned)(own >> 5)) + off);
      mask_count<P, MODE == EVAL_INIT_CN>(a.masks, off, nn, cnt);
      if (MODE == EVAL_REFINE) lg += (int)__popcll(__ballot(((sw >> (own & 31)) & 1u) != 0u));
    };
    if (WIDE && deg > MASK_WIDE) {
      mask_count_wide<P>(masks, nets, vb, deg, (unsigned)a.noe * ROW, s_wide[WIDE ? wave : 0], cnt, [&](unsigned off) {
        if (MODE != EVAL_REFINE) return;
        const unsigned sw = *reinterpret_cast<const unsigned*>(masks + (8u * P + 4u * (unsigned)(own >> 5)) + off);
        lg += (int)__popcll(__ballot(((sw >> (own & 31)) & 1u) != 0u));
      });
      load_parts();  // so that their registers are free above
    } else {
      count_nets(id0, min(deg, CH));
      for (int c0 = CH; c0 < deg; c0 += CH)
        count_nets(*reinterpret_cast<const unsigned*>(nets + min(vb + (unsigned)(c0 + lane), a.last_pin) * 4u),
                   min(deg - c0, CH));
    }
    unsigned craw = 0;
    const int pl = mask_ldg<P, MODE == EVAL_INIT_CN>(a.masks, a.vtx_nets, a.vtx_seg, a.ev, vb, deg,
                                                     MODE == EVAL_REFINE ? own : -1, cnt, pen, skey, pid, craw);
    int d = pl < 0 ? -1 : pl & 0xFFFF;
    bool in_band = pl >= 0 && (pl >> 16) != 0;
    const bool none = d < 0;  // no part above score 0: the fallback
    int dd;
    if (MODE == EVAL_REFINE) {
      if (none) {
        d = wave_lightest_part(a.sizes, K);
        int px = 0;
        unsigned cx = 0;
#pragma unroll
        for (int u = 0; u < P; u++) {
          px = (d >> 6) == u ? pid[u] : px;
          cx = (d >> 6) == u ? cnt[u] : cx;
        }
        in_band = (__builtin_amdgcn_readlane(px, d & (WAVE - 1)) >> 16) != 0;
        craw = (unsigned)__builtin_amdgcn_readlane((int)cx, d & (WAVE - 1)) - MASK_BIAS;
      }
      // outside the bands the vertex stays (TV/partition.cpp:135-143)
      const int al = deg - (int)craw;  // arrival loss: nets of v lacking d (TV/partition.cpp:369-377)
      const bool accept = in_band && d != own && lg >= al;  // TV/partition.cpp:380
      dd = accept ? d : -1;
      if (accept && a.net_stamp) {
        if (lane < min(deg, CH)) a.net_stamp[id0] = a.tag;
        if (deg > CH) wave_stamp_nets(a.vtx_nets + (vb + (unsigned)CH), deg - CH, a.tag, a.net_stamp);
      }
    } else {
      // an unplaced vertex with no part above score 0, or whose choice is
      // above the band, takes its turn in the fallback
      dd = none || !in_band ? SLOT_FALLBACK : d;
    }
    dec_l = lane == i ? dd : dec_l;
  }
  if (lane < ns) {
    a.slot_own[slot_l] = own_l;
    a.slot_dec[slot_l] = dec_l;
    if (dec_l >= 0 && a.hist) {
      const int w = a.vwgt ? a.vwgt[v_l] : 1;
      atomicAdd(&a.hist[(size_t)dec_l * (size_t)a.ntiles + (size_t)(slot_l / TILE)], w);
    }
  }
}

// the instance of k_tv_eval_masks for K parts
template <int MODE>
void (*eval_masks_kernel(int K, bool wide))(EvalArgs) {
  if constexpr (MODE != EVAL_INIT_CN) {
    if (wide) switch (mask_words(K)) {
        case 5: return k_tv_eval_masks<5, MODE, true>;
        case 6: return k_tv_eval_masks<6, MODE, true>;
        case 7: return k_tv_eval_masks<7, MODE, true>;
        default: return k_tv_eval_masks<8, MODE, true>;
      }
  }
  switch (mask_words(K)) {
    case 1: return k_tv_eval_masks<1, MODE, false>;
    case 2: return k_tv_eval_masks<2, MODE, false>;
    case 3: return k_tv_eval_masks<3, MODE, false>;
    case 4: return k_tv_eval_masks<4, MODE, false>;
    case 5: return k_tv_eval_masks<5, MODE, false>;
    case 6: return k_tv_eval_masks<6, MODE, false>;
    case 7: return k_tv_eval_masks<7, MODE, false>;
    default: return k_tv_eval_masks<8, MODE, false>;
  }
}

// BAL step 1, per part: its candidates' weight is its row of the tile
// histogram. A part whose candidates exceed cap - size is over-subscribed:
// over[d] is set and pref's row d receives the exclusive prefix sums of the
// tiles. The row is cleared for the next round. Rows of up to
// SCAN_WAVE_TILES tiles are taken by one wavefront each, longer ones by a block,
// whose threads load SCAN_RUN consecutive tiles together: a 4096-tile row
// takes one round trip to memory and one block scan. Summing the rows here
// spares the evaluation a 64-bit atomic per candidate on one of K words.
constexpr int SCAN_WAVE_TILES = 16 * WAVE;

template <bool WAVE_ROWS>
__global__ void __launch_bounds__(256) k_bal_scan(int* __restrict__ hist, long long* __restrict__ pref, int ntiles,
                                                  int K, const long long* __restrict__ sizes_frozen, long long cap,
                                                  int* __restrict__ over, int* __restrict__ tcount) {
  __shared__ long long s_wl[16];
  const int lane = lane_id();
  if (blockIdx.x == 0 && threadIdx.x == 0) *tcount = 0;  // of the round's touched list (k_bal_admit)
  if (WAVE_ROWS) {
    const int nw = (int)(blockDim.x / WAVE);
    for (int d = (int)blockIdx.x * nw + wave_id(); d < K; d += (int)gridDim.x * nw) {
      int* row = hist + (size_t)d * (size_t)ntiles;
      int x[SCAN_WAVE_TILES / WAVE];
      int sum = 0;  // total weights fit an int
#pragma unroll
      for (int p = 0; p < SCAN_WAVE_TILES / WAVE; p++) {
        const int t = p * WAVE + lane;
        x[p] = t < ntiles ? row[t] : 0;
      }
#pragma unroll
      for (int p = 0; p < SCAN_WAVE_TILES / WAVE; p++) sum += x[p];
      const int tot = wave_sum(sum);
      const bool ov = tot > cap - sizes_frozen[d];
      if (lane == 0) over[d] = ov ? 1 : 0;
      if (tot == 0 && !ov) continue;
      int acc = 0;
#pragma unroll
      for (int p = 0; p < SCAN_WAVE_TILES / WAVE; p++) {
        const int t = p * WAVE + lane;
        if (ov && p * WAVE < ntiles) {
          const int incl = wave_incl_scan(x[p]);
          if (t < ntiles) pref[(size_t)d * (size_t)ntiles + (size_t)t] = acc + (incl - x[p]);
          acc += __builtin_amdgcn_readlane(incl, WAVE - 1);
        }
        if (t < ntiles && x[p]) row[t] = 0;
      }
    }
    return;
  }
  const int step = (int)blockDim.x * SCAN_RUN;
  for (int d = (int)blockIdx.x; d < K; d += (int)gridDim.x) {
    int* row = hist + (size_t)d * (size_t)ntiles;
    long long* out = pref + (size_t)d * (size_t)ntiles;
    int x[SCAN_RUN];
    auto load = [&](int t0) -> long long {
      const int tb = t0 + (int)threadIdx.x * SCAN_RUN;
      long long run = 0;
#pragma unroll
      for (int p = 0; p < SCAN_RUN; p++) {
        const int v = row[min(tb + p, ntiles - 1)];
        x[p] = tb + p < ntiles ? v : 0;
      }
#pragma unroll
      for (int p = 0; p < SCAN_RUN; p++) run += x[p];
      return run;
    };
    long long sum = 0, first = 0;
    for (int t0 = 0; t0 < ntiles; t0 += step) {
      const long long r = load(t0);
      if (t0 == 0) first = r;
      sum += r;
    }
    long long tot;
    (void)block_excl_scan(sum, s_wl, &tot);
    const bool ov = tot > cap - sizes_frozen[d];
    if (threadIdx.x == 0) over[d] = ov ? 1 : 0;
    if (tot == 0 && !ov) continue;
    long long carry = 0;
    for (int t0 = 0; t0 < ntiles; t0 += step) {
      const long long run = ntiles > step ? load(t0) : first;
      const int tb = t0 + (int)threadIdx.x * SCAN_RUN;
      if (ov) {
        long long chunk;
        long long acc = carry + block_excl_scan(run, s_wl, &chunk);
#pragma unroll
        for (int p = 0; p < SCAN_RUN; p++) {
          if (tb + p < ntiles) out[tb + p] = acc;
          acc += x[p];
        }
        carry += chunk;
      }
#pragma unroll
      for (int p = 0; p < SCAN_RUN; p++)
        if (tb + p < ntiles && x[p]) row[tb + p] = 0;
    }
  }
}

// Initial partition, between the evaluation and the admission (one block):
// the j-th fallback slot of the sub-round, in slot order, takes part
// (fb + j) mod K, fb the lowest-index part of minimum frozen size, and its
// weight joins the tile histogram.
constexpr int FALLBACK_RUN = 16;  // consecutive slots per thread in k_init_fallback

__global__ void __launch_bounds__(1024) k_init_fallback(int* __restrict__ slot_dec, const int* __restrict__ order,
                                                        const int* __restrict__ vwgt, int r0, int nslots, int ntiles,
                                                        int K, const int* __restrict__ fb_in, int* __restrict__ hist) {
  __shared__ int s_wi[16];
  const int fb = *fb_in;
  int carry = 0;
  // each thread takes FALLBACK_RUN consecutive slots, their decisions loaded
  // together: a sub-round of 16,384 slots is one load round trip and one
  // block scan
  for (int b0 = 0; b0 < nslots; b0 += (int)blockDim.x * FALLBACK_RUN) {
    const int base = b0 + (int)threadIdx.x * FALLBACK_RUN;
    int dec[FALLBACK_RUN];
#pragma unroll
    for (int q = 0; q < FALLBACK_RUN; q++) dec[q] = base + q < nslots ? slot_dec[base + q] : 0;
    int cnt = 0;
#pragma unroll
    for (int q = 0; q < FALLBACK_RUN; q++) cnt += dec[q] == SLOT_FALLBACK ? 1 : 0;
    int tot;
    int j = carry + block_excl_scan(cnt, s_wi, &tot);
    if (cnt)
      for (int q = 0; q < FALLBACK_RUN; q++) {
        if (dec[q] != SLOT_FALLBACK) continue;
        const int slot = base + q;
        const int d = (int)(((long long)fb + j) % K);
        j++;
        slot_dec[slot] = d;
        const int z = r0 + slot;
        const int w = vwgt ? vwgt[order ? order[z] : z] : 1;
        atomicAdd(&hist[(size_t)d * (size_t)ntiles + (size_t)(slot / TILE)], w);
      }
    carry += tot;
  }
}

// BAL step 2, one wavefront per tile: a candidate into an over-subscribed part
// d is admitted iff frozen_size[d] + (weight of earlier candidates into d) + w
// <= cap (first_free: or it is the first candidate into d); every other
// candidate is admitted. Commits part vector and sizes of admitted moves (a
// vertex without a part, own -1, only adds to its new part's size). AGG:
// the block sums its size changes per part in LDS first, so that sizes takes
// one atomic per part and block (same-address atomics from every wave would
// queue at one L2 slice, about 12 ns each).
constexpr int ADMIT_BLOCK = 512;
constexpr int ADMIT_NETS = 4;

// LIST: the touched nets go to a list, too (apply_by_list).
template <bool AGG, bool LIST>
__global__ void __launch_bounds__(ADMIT_BLOCK) k_bal_admit(int* __restrict__ slot_dec, const int* __restrict__ slot_own,
                                                   const int* __restrict__ order, const int* __restrict__ vwgt,
                                                   int r0, int nslots, int ntiles, int K,
                                                   const long long* __restrict__ sizes_frozen, long long cap,
                                                   bool first_free, const int* __restrict__ over,
                                                   const long long* __restrict__ pref, int* __restrict__ part,
                                                   long long* __restrict__ sizes,
                                                   unsigned long long* __restrict__ moves,
                                                   const unsigned* __restrict__ vtx_ptr,
                                                   const unsigned* __restrict__ vtx_nets, unsigned tag,
                                                   unsigned* __restrict__ net_stamp, int* __restrict__ touched,
                                                   int* __restrict__ tcount) {
  const int lane = lane_id(), wave = wave_id(), nw = (int)(blockDim.x / WAVE);
  // the block's admitted moves, added to the global count once per block
  // (same-address atomics from every wave would queue at one L2 slice)
  __shared__ unsigned long long s_moves;
  // AGG: the block's size changes per part, added to sizes once per block
  extern __shared__ __align__(16) unsigned char lds[];
  unsigned long long* s_dsz = reinterpret_cast<unsigned long long*>(lds);
  if (threadIdx.x == 0) s_moves = 0;
  if (AGG)
    for (int d = (int)threadIdx.x; d < K; d += (int)blockDim.x) s_dsz[d] = 0;
  __syncthreads();
  for (int tile = (int)blockIdx.x * nw + wave; tile < ntiles; tile += (int)gridDim.x * nw) {
    const int slot = tile * TILE + lane;
    int d = -1, v = -1;
    long long w = 0;
    unsigned vb = 0, ve = 0;
    if (slot < nslots) {
      d = slot_dec[slot];
      const int z = r0 + slot;
      v = order ? order[z] : z;
      w = vwgt ? vwgt[v] : 1;
      if (LIST) {
        // of the stream, whose candidates are nearly all admitted, and whose
        // small launches are a chain of loads
        vb = vtx_ptr[v];
        ve = vtx_ptr[v + 1];
      }
    }
    unsigned n[ADMIT_NETS];
    if (LIST && d >= 0 && vb < ve) {
#pragma unroll
      for (int u = 0; u < ADMIT_NETS; u++) n[u] = vtx_nets[min(vb + (unsigned)u, ve - 1)];
    }
    const bool o = d >= 0 && over[d] != 0;
    bool adm = d >= 0;
    if (__ballot(o)) {
      // weight of earlier candidates into the same part within the tile
      long long pre = 0;
      const int wi = (int)w;  // vertex weights are int
      for (int j = 0; j < WAVE; j++) {
        const int dj = __builtin_amdgcn_readlane(d, j), wj = __builtin_amdgcn_readlane(wi, j);
        if (j < lane && dj == d) pre += wj;
      }
      if (o) {
        const long long before = pref[(size_t)d * (size_t)ntiles + (size_t)tile] + pre;
        adm = sizes_frozen[d] + before + w <= cap || (first_free && before == 0);
      }
    }
    if (d >= 0 && !adm) slot_dec[slot] = -1;
    if (adm) {
      part[v] = d;
      const int own = slot_own[slot];
      if (AGG) {
        if (own >= 0) atomicAdd(&s_dsz[own], (unsigned long long)-w);
        atomicAdd(&s_dsz[d], (unsigned long long)w);
      } else {
        if (own >= 0) atomic_add_i64(&sizes[own], -w);
        atomic_add_i64(&sizes[d], w);
      }
    }
    // the admitted moves' nets get the round's tag: by the move's lane,
    // ADMIT_NETS at a time, or by the wave for a vertex of more than 64 nets
    if (!LIST && adm) {
      vb = vtx_ptr[v];
      ve = vtx_ptr[v + 1];
    }
    const bool hub = adm && ve - vb > (unsigned)WAVE;
    unsigned long long fresh = 0;  // LIST, bit j: the lane stamped its net j first
    if (adm && !hub)
      for (unsigned j = vb; j < ve; j += ADMIT_NETS) {
        // past the end the last net again (LIST: it has the tag by then)
        if (!LIST || j != vb) {
#pragma unroll
          for (int u = 0; u < ADMIT_NETS; u++) n[u] = vtx_nets[min(j + (unsigned)u, ve - 1)];
        }
        if (!LIST) {
#pragma unroll
          for (int u = 0; u < ADMIT_NETS; u++) net_stamp[n[u]] = tag;
        } else {
          unsigned old[ADMIT_NETS];
#pragma unroll
          for (int u = 0; u < ADMIT_NETS; u++) old[u] = atomicExch(&net_stamp[n[u]], tag);
#pragma unroll
          for (int u = 0; u < ADMIT_NETS; u++) fresh |= old[u] != tag ? 1ull << (j - vb + (unsigned)u) : 0ull;
        }
      }
    if (LIST) {
      const int mine = (int)__popcll(fresh), incl = wave_incl_scan(mine);
      const int all = __builtin_amdgcn_readlane(incl, WAVE - 1);
      int at = 0;
      if (all && lane == 0) at = atomicAdd(tcount, all);
      at = __builtin_amdgcn_readlane(at, 0) + incl - mine;
      for (; fresh; fresh &= fresh - 1) touched[at++] = (int)vtx_nets[vb + (unsigned)__builtin_ctzll(fresh)];
    }
    for (unsigned long long hm = __ballot(hub); hm; hm &= hm - 1) {
      const int l = __ffsll((long long)hm) - 1;
      const unsigned b = (unsigned)__builtin_amdgcn_readlane((int)vb, l), e = (unsigned)__builtin_amdgcn_readlane((int)ve, l);
      if (!LIST) {
        wave_stamp_nets(vtx_nets + b, (int)(e - b), tag, net_stamp);
        continue;
      }
      for (unsigned j = b; j < e; j += (unsigned)WAVE) {
        unsigned n = 0;
        bool first = false;
        if (j + (unsigned)lane < e) {
          n = vtx_nets[j + (unsigned)lane];
          first = atomicExch(&net_stamp[n], tag) != tag;
        }
        const unsigned long long fm = __ballot(first);
        int at = 0;
        if (fm && lane == 0) at = atomicAdd(tcount, (int)__popcll(fm));
        at = __builtin_amdgcn_readlane(at, 0);
        if (first) touched[at + (int)__popcll(fm & ((1ull << lane) - 1ull))] = (int)n;
      }
    }
    const unsigned long long am = __ballot(adm);
    if (lane == 0 && am) atomicAdd(&s_moves, (unsigned long long)__popcll(am));
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_moves) atomicAdd(moves, s_moves);
  if (AGG)
    for (int d = (int)threadIdx.x; d < K; d += (int)blockDim.x) {
      const long long x = (long long)s_dsz[d];
      if (x) atomic_add_i64(&sizes[d], x);
    }
}

struct ApplyArgs {
  const unsigned* net_ptr;
  const int* apply_pins;
  const int* slot_own;
  const int* slot_dec;
  const unsigned* net_stamp;  // the nets stamped with the round's tag are touched
  unsigned tag;
  int noe, per_block;         // each block takes per_block consecutive nets
  const int* touched;         // LIST: the touched nets, shared by the blocks
  const int* tcount;
  int lane_words;             // LDS words per lane of the small nets' replay
  int wave_bytes;             // LDS bytes per wave
  unsigned* ent;
  unsigned short* ev;
  unsigned long long* masks;  // nullable: the nets' part masks, kept in step with the lists
  int mask_words;
  int K, pb;
  unsigned pmask;
  int r0, r1;
  // REF commit in blocks >= net_blocks (nullable part: no commit)
  int net_blocks;
  const int* order;
  int* part;
  long long* sizes;
  unsigned long long* moves;
};

// One lane replays the round's moves on a net of at most SMALL_NET pins, in
// the rank order of its pins, on a copy of the list in its registers: the
// same edits, in the same order, as the wavefront replay (remove = decrement
// or swap-with-last, add = increment or append). The list and the ranks load
// together, then the moves of the ranked pins. A list in the lane's LDS words
// instead waited out an LDS read per entry looked at (13 to 25 us for 64 nets).
__device__ __forceinline__ void lane_replay_small(const ApplyArgs& a, int n, unsigned s, unsigned np, unsigned* my) {
  const unsigned seg = s + (unsigned)n;
  int r[SMALL_NET];
  unsigned x[SMALL_NET + 1];
#pragma unroll
  for (int i = 0; i < SMALL_NET; i++) r[i] = (unsigned)i < np ? a.apply_pins[s + (unsigned)i] : INT_MAX;
#pragma unroll
  for (int t = 0; t <= SMALL_NET; t++) x[t] = (unsigned)t <= np ? a.ent[seg + (unsigned)t] : 0u;
  int dd[SMALL_NET], oo[SMALL_NET];
#pragma unroll
  for (int i = 0; i < SMALL_NET; i++) {
    const bool in = r[i] >= a.r0 && r[i] < a.r1;
    dd[i] = in ? a.slot_dec[r[i] - a.r0] : -1;
    oo[i] = in ? a.slot_own[r[i] - a.r0] : -1;
  }
  int L = (int)x[0];
  int key[SMALL_NET];  // part of each entry, -1 past the list
  int cnt[SMALL_NET];
#pragma unroll
  for (int t = 0; t < SMALL_NET; t++) {
    key[t] = t < L ? (int)(x[t + 1] & a.pmask) : -1;
    cnt[t] = (int)(x[t + 1] >> a.pb);
  }
  bool any = false;
#pragma unroll
  for (int i = 0; i < SMALL_NET; i++) {
    if (dd[i] < 0) continue;
    any = true;
    const int p = oo[i], q = dd[i];
    // the last entry, should it have to fill p's place
    int lk = -1, lc = 0;
#pragma unroll
    for (int t = 0; t < SMALL_NET; t++) {
      lk = t == L - 1 ? key[t] : lk;
      lc = t == L - 1 ? cnt[t] : lc;
    }
    bool gone = false;
#pragma unroll
    for (int t = 0; t < SMALL_NET; t++) {
      const bool hit = p >= 0 && key[t] == p;
      const bool last = hit && cnt[t] == 1;
      gone |= last;
      key[t] = last ? lk : key[t];
      cnt[t] = last ? lc : cnt[t] - (hit ? 1 : 0);
    }
    L -= gone ? 1 : 0;
    bool found = false;
#pragma unroll
    for (int t = 0; t < SMALL_NET; t++) {
      key[t] = gone && t == L ? -1 : key[t];
      const bool hit = key[t] == q;
      found |= hit;
      cnt[t] += hit ? 1 : 0;
    }
#pragma unroll
    for (int t = 0; t < SMALL_NET; t++) {
      key[t] = !found && t == L ? q : key[t];
      cnt[t] = !found && t == L ? 1 : cnt[t];
    }
    L += found ? 0 : 1;
  }
  if (!any) return;
  unsigned y[SMALL_NET];
#pragma unroll
  for (int t = 0; t < SMALL_NET; t++) {
    y[t] = ((unsigned)cnt[t] << a.pb) | (unsigned)key[t];
    if (t < L) {
      a.ent[seg + 1 + (unsigned)t] = y[t];
      a.ev[seg + 1 + (unsigned)t] = ev_word(y[t], a.pb, a.pmask);
    }
  }
  a.ent[seg] = (unsigned)L;
  a.ev[seg] = (unsigned short)L;
  if (a.masks) lane_store_masks(y, L, a.pb, a.pmask, a.mask_words, my, a.masks + (size_t)n * (size_t)(2 * a.mask_words));
}

// One wavefront replays the round's moves (lane l: dd >= 0, the part its pin
// moves to, and oo, the part it leaves) on a net of at most 64 pins, lane t
// holding entry t of the list: an edit is a few ballots and lane writes, with
// no LDS.
__device__ __forceinline__ void wave_replay_medium(const ApplyArgs& a, int n, unsigned s, int L0, unsigned x, int dd,
                                                   int oo, unsigned* words) {
  const int lane = lane_id();
  const unsigned seg = s + (unsigned)n;
  int L = L0;
  int key = lane < L ? (int)(x & a.pmask) : -1;
  unsigned cnt = x >> a.pb;
  for (unsigned long long m = __ballot(dd >= 0); m; m &= m - 1) {
    const int l = __ffsll((long long)m) - 1;
    const int p = __builtin_amdgcn_readlane(oo, l), q = __builtin_amdgcn_readlane(dd, l);
    const unsigned long long mp = __ballot(key == p && p >= 0);
    if (mp) {
      const int jp = __ffsll((long long)mp) - 1;
      if (__builtin_amdgcn_readlane((int)cnt, jp) > 1) {
        cnt -= key == p ? 1u : 0u;
      } else {
        // the last entry takes p's place
        L--;
        const int lk = __builtin_amdgcn_readlane(key, L), lc = __builtin_amdgcn_readlane((int)cnt, L);
        key = lane == jp ? lk : key;
        cnt = lane == jp ? (unsigned)lc : cnt;
        key = lane == L ? -1 : key;
      }
    }
    const unsigned long long mq = __ballot(key == q);
    if (mq) {
      cnt += key == q ? 1u : 0u;
    } else {
      key = lane == L ? q : key;
      cnt = lane == L ? 1u : cnt;
      L++;
    }
  }
  const unsigned y = (cnt << a.pb) | (unsigned)key;
  if (lane < L) {
    a.ent[seg + 1 + (unsigned)lane] = y;
    a.ev[seg + 1 + (unsigned)lane] = ev_word(y, a.pb, a.pmask);
  }
  if (lane == 0) {
    a.ent[seg] = (unsigned)L;
    a.ev[seg] = (unsigned short)L;
  }
  if (a.masks) wave_store_entry_masks(lane < L, (unsigned)key, cnt, a.mask_words, words,
                                      a.masks + (size_t)n * (size_t)(2 * a.mask_words));
}

// The apply's LDS that does not depend on K: the block's touched nets (the
// small ones from the front, the others from the back), the positions of the
// huge ones, which are replayed first, and the waves' mask words.
template <bool LIST>
struct ApplyNets {
  int cnt[4];  // touched small nets, other nets, nets handed out, huge nets
  unsigned words[APPLY_BLOCK / WAVE][4 * MASK_PMAX];
  unsigned start[APPLY_NETS], len[APPLY_NETS];
  std::conditional_t<LIST, unsigned, unsigned short> net[APPLY_NETS];  // LIST: its number, else from the block's first net on
  unsigned short huge[APPLY_NETS];
};

// Replays the round's moves on every touched net in ordering order
// (TV/partition.cpp:846-890: remove = decrement or swap-with-last, add =
// increment or append): a lane per small net, a wavefront per other one.
// Blocks past net_blocks commit the REF part vector and source-part sizes
// (TV/partition.cpp:818-830: the destination's size is left unchanged).
// INDEXED: each wave keeps a part -> position index of its list in LDS (2
// bytes per part after the list), for K where it fits.
// LIST: the touched nets come as a list, else each block looks for them among
// the stamps of its nets (apply_by_list).
template <bool INDEXED, bool LIST>
__global__ void __launch_bounds__(APPLY_BLOCK) __attribute__((amdgpu_waves_per_eu(8))) k_apply(ApplyArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int lane = lane_id(), wave = wave_id(), nw = (int)(blockDim.x / WAVE);
  if ((int)blockIdx.x >= a.net_blocks) {
    const int slot = ((int)blockIdx.x - a.net_blocks) * (int)blockDim.x + (int)threadIdx.x;
    bool mv = false;
    if (slot < a.r1 - a.r0) {
      const int d = a.slot_dec[slot];
      if (d >= 0) {
        const int z = a.r0 + slot;
        a.part[a.order ? a.order[z] : z] = d;
        atomic_add_i64(&a.sizes[a.slot_own[slot]], -1);
        mv = true;
      }
    }
    block_count_add(a.moves, mv);
    return;
  }
  // the wave's own region: first the lanes' words of their mask records (an
  // odd number each, which keeps them on distinct banks), then a net's
  unsigned char* mem = lds + (size_t)wave * (size_t)a.wave_bytes;
  unsigned* my = reinterpret_cast<unsigned*>(mem) + (size_t)lane * (size_t)a.lane_words;
  unsigned* list = reinterpret_cast<unsigned*>(mem);
  unsigned short* at = reinterpret_cast<unsigned short*>(list + a.K);
  __shared__ ApplyNets<LIST> s;
  unsigned* words = s.words[wave];

  // the block's touched nets, the small ones and the others apart: a wave
  // then replays 64 small nets at a time, a lane each, and the big ones go
  // to whichever wave is free
  const int total = LIST ? *a.tcount : a.noe;
  const int per = LIST ? min(APPLY_NETS, max(APPLY_LIST_NETS, (total + a.net_blocks - 1) / a.net_blocks)) : a.per_block;
  const int n0 = (int)blockIdx.x * per, net0 = LIST ? 0 : n0;
  const int nn = min(per, total - n0);
  if (LIST && nn <= 0) return;
  if (threadIdx.x < 4) s.cnt[threadIdx.x] = 0;
  __syncthreads();
  // the stamps (or numbers) of all the thread's nets load together, then their pin ranges
  constexpr int OWN = APPLY_NETS / APPLY_BLOCK;
  unsigned net[OWN], first[OWN], last[OWN];
#pragma unroll
  for (int u = 0; u < OWN; u++) {
    const int i = u * APPLY_BLOCK + (int)threadIdx.x;
    net[u] = i < nn ? (LIST ? (unsigned)a.touched[n0 + i] : a.net_stamp[n0 + i]) : ~0u;
  }
#pragma unroll
  for (int u = 0; u < OWN; u++) {
    const int i = u * APPLY_BLOCK + (int)threadIdx.x;
    const bool hit = i < nn && (LIST || net[u] == a.tag);
    net[u] = hit ? (LIST ? net[u] : (unsigned)(n0 + i)) : ~0u;
    first[u] = last[u] = 0;
    if (hit) {
      first[u] = a.net_ptr[net[u]];
      last[u] = a.net_ptr[net[u] + 1];
    }
  }
#pragma unroll
  for (int u = 0; u < OWN; u++) {
    const unsigned n = net[u], st = first[u], len = last[u] - first[u];
    const bool hit = n != ~0u;
    const bool sm = hit && len <= (unsigned)SMALL_NET;
    const unsigned long long ms = __ballot(sm), mb = __ballot(hit && !sm);
    int bs = 0, bb = 0;
    if (lane == 0) {
      if (ms) bs = atomicAdd(&s.cnt[0], (int)__popcll(ms));
      if (mb) bb = atomicAdd(&s.cnt[1], (int)__popcll(mb));
    }
    // lane 0's, read while every lane is active
    bs = __builtin_amdgcn_readlane(bs, 0);
    bb = __builtin_amdgcn_readlane(bb, 0);
    const unsigned long long lt = (1ull << lane) - 1ull;
    const int k = sm ? bs + (int)__popcll(ms & lt) : APPLY_NETS - 1 - (bb + (int)__popcll(mb & lt));
    if (hit) {
      s.net[k] = (decltype(s.net[0] + 0))(n - (unsigned)net0);
      s.start[k] = st;
      s.len[k] = len;
      if (len >= HUGE_NET) s.huge[atomicAdd(&s.cnt[3], 1)] = (unsigned short)k;
    }
  }
  __syncthreads();
  const int nsmall = __builtin_amdgcn_readfirstlane(s.cnt[0]), nbig = __builtin_amdgcn_readfirstlane(s.cnt[1]);
  const int nhuge = __builtin_amdgcn_readfirstlane(s.cnt[3]);

  for (int b = wave * WAVE; b < nsmall; b += nw * WAVE)
    if (b + lane < nsmall) lane_replay_small(a, net0 + (int)s.net[b + lane], s.start[b + lane], s.len[b + lane], my);
  if (nbig == 0) return;
  wave_lds_sync();
  if (INDEXED) wave_index_init(at, a.K);

  // The others in three stages, so that a net of at most 64 pins waits for no
  // load of its own: its head (its list and its ranks; of a larger net the
  // first 64 words of its segment) loads while the net before the previous
  // one is replayed, its ranks' decisions while the previous one is
  struct NetHead {
    int n, r, dd, oo, L;
    unsigned s, e, x;
  };
  auto next_head = [&]() -> NetHead {
    NetHead h{-1, INT_MAX, -1, -1, 0, 0u, 0u, 0u};
    int k = 0;
    if (lane == 0) k = atomicAdd(&s.cnt[2], 1);
    k = __builtin_amdgcn_readlane(k, 0);
    for (;;) {
      if (k >= nhuge + nbig) return h;
      if (k < nhuge) {
        k = __builtin_amdgcn_readfirstlane((int)s.huge[k]);
        break;
      }
      k = APPLY_NETS - 1 - (k - nhuge);
      if (nhuge == 0 || __builtin_amdgcn_readfirstlane((int)s.len[k]) < (int)HUGE_NET) break;
      if (lane == 0) k = atomicAdd(&s.cnt[2], 1);  // a huge one again: the next
      k = __builtin_amdgcn_readlane(k, 0);
    }
    h.n = net0 + __builtin_amdgcn_readfirstlane((int)s.net[k]);
    h.s = (unsigned)__builtin_amdgcn_readfirstlane((int)s.start[k]);
    const unsigned np = (unsigned)__builtin_amdgcn_readfirstlane((int)s.len[k]);
    h.e = h.s + np;
    const unsigned seg = h.s + (unsigned)h.n;
    if (np <= (unsigned)WAVE) {
      h.L = (int)a.ent[seg];
      h.x = (unsigned)lane < np ? a.ent[seg + 1u + (unsigned)lane] : 0u;
      h.r = (unsigned)lane < np ? a.apply_pins[h.s + (unsigned)lane] : INT_MAX;
    } else {
      h.x = wave_list_head(a.ent, seg, np);
    }
    return h;
  };
  auto load_moves = [&](NetHead& h) {
    if (h.r >= a.r0 && h.r < a.r1) {
      h.dd = a.slot_dec[h.r - a.r0];
      h.oo = a.slot_own[h.r - a.r0];
    }
  };
  auto replay_net = [&](const NetHead& h) {
    const int n = h.n;
    const unsigned b = h.s, e = h.e;
    const unsigned seg = b + (unsigned)n;
    if (e - b <= (unsigned)WAVE) {
      if (__ballot(h.dd >= 0)) wave_replay_medium(a, n, b, __builtin_amdgcn_readfirstlane(h.L), h.x, h.dd, h.oo, words);
      return;
    }
    unsigned lo, hi;
    wave_rank_window(a.apply_pins, b, e, a.r0, a.r1, lo, hi);
    int L = wave_list_stage(a.ent, seg, h.x, list);
    if (INDEXED) wave_index_set(list, L, at, a.pmask);
    bool dirty = false;
    // the round's pins of the net, APPLY_GROUP windows of 64 ranks at a time:
    // their ranks load together, then their slots' decisions, so that a big
    // net (a Zipf net of thousands of pins, a quarter of them in the round)
    // takes a few dependent load rounds instead of one per window
    for (unsigned k0 = lo; k0 < hi; k0 += APPLY_GROUP * WAVE) {
      int rr[APPLY_GROUP], dd[APPLY_GROUP], oo[APPLY_GROUP];
#pragma unroll
      for (int u = 0; u < APPLY_GROUP; u++) {
        const unsigned k = k0 + (unsigned)(u * WAVE + lane);
        rr[u] = k < hi ? a.apply_pins[k] : INT_MAX;
      }
#pragma unroll
      for (int u = 0; u < APPLY_GROUP; u++) {
        dd[u] = -1;
        oo[u] = -1;
        if (rr[u] >= a.r0 && rr[u] < a.r1) {
          dd[u] = a.slot_dec[rr[u] - a.r0];
          oo[u] = a.slot_own[rr[u] - a.r0];
        }
      }
#pragma unroll
      for (int u = 0; u < APPLY_GROUP; u++) {
        unsigned long long m = __ballot(dd[u] >= 0);
        dirty |= m != 0;
        if (INDEXED && m && __ballot(dd[u] >= 0 && oo[u] >= 0) == 0ull) {
          wave_ilist_places(list, at, L, m, dd[u], a.pb);
          continue;
        }
        bool together = INDEXED;  // worth trying in this window
        while (m) {
          if (together && __popcll(m) >= APPLY_TOGETHER) {
            const int before = (int)__popcll(m);
            m = wave_ilist_moves(list, at, m, oo[u], dd[u], a.pb);
            together = before - (int)__popcll(m) >= APPLY_TOGETHER / 2;
            if (!m) break;
          }
          const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)m) - 1);
          m &= m - 1;
          const int o = __builtin_amdgcn_readlane(oo[u], l), d = __builtin_amdgcn_readlane(dd[u], l);
          if (INDEXED) {
            unsigned co;
            bool found;
            wave_ilist_move(list, at, L, o, d, a.pb, a.pmask, co, found);
          } else {
            wave_list_move(list, L, o, d, a.pb, a.pmask);
          }
        }
      }
    }
    if (dirty) wave_list_store(a.ent, a.ev, seg, list, L, a.pb, a.pmask);
    if (INDEXED && dirty && a.masks)
      wave_store_masks(list, at, a.K, a.pb, a.mask_words, a.masks + (size_t)n * (size_t)(2 * a.mask_words));
    if (INDEXED) wave_index_clear(list, L, at, a.pmask);
    wave_lds_sync();
  };
  NetHead cur = next_head(), nxt = next_head();
  load_moves(cur);
  while (cur.n >= 0) {
    const NetHead nn2 = next_head();
    load_moves(nxt);
    replay_net(cur);
    cur = nxt;
    nxt = nn2;
  }
}

// LDS of the apply, per wave: a K-entry list and, where it fits the budget,
// the part -> position index, or before that half a mask record per lane
int apply_lane_words(int K) { return 2 * mask_words(K) + 1; }

size_t apply_wave_bytes(int K, bool indexed) {
  const size_t list = (size_t)K * (sizeof(unsigned) + (indexed ? sizeof(unsigned short) : 0));
  return (std::max(list, (size_t)WAVE * (size_t)apply_lane_words(K) * sizeof(unsigned)) + 15) & ~(size_t)15;
}

size_t apply_static(bool list) { return list ? sizeof(ApplyNets<true>) : sizeof(ApplyNets<false>); }

bool apply_indexed(int K, bool list) {
  return (size_t)(APPLY_BLOCK / WAVE) * apply_wave_bytes(K, true) + apply_static(list) <= (size_t)LDS_BUDGET;
}

size_t apply_lds(int K, bool list) { return (size_t)(APPLY_BLOCK / WAVE) * apply_wave_bytes(K, apply_indexed(K, list)); }

size_t eval_lds(int K, int waves) {
  return (size_t)K * 12 + (size_t)waves * 8 * (size_t)(K + WAVE);
}

// the largest K of the refinements with a schedule and of the device stream:
// 12 + 8 bytes per part and 1.5 KiB in one workgroup of one wavefront
constexpr int EVAL_KMAX = (LDS_BUDGET - 1536) / 20;

int eval_waves(int K) {
  // LDS: 12 bytes per part shared by the block + 8 bytes per part (and per
  // spare slot) per wavefront
  if (K > EVAL_KMAX) return 0;
  for (int w = EVAL_BLOCK / WAVE; w >= 1; w--)
    if (eval_lds(K, w) <= (size_t)LDS_BUDGET) return w;
  return 0;
}

int eval_grid(int nslots, int waves) { return std::max(1, std::min((nslots + waves - 1) / waves, 8192)); }

fp_status ensure_round_scratch(fp_ctx* ctx, int R) {
  if (R > ctx->rmax) {
    FP_TRY(dalloc(ctx, &ctx->slot_own, (size_t)R));
    FP_TRY(dalloc(ctx, &ctx->slot_dec, (size_t)R));
    ctx->rmax = R;
  }
  return FP_OK;
}

// of ensure_bal_scratch: an int and a long long per part and tile
constexpr long long BAL_BYTES = sizeof(int) + sizeof(long long);

fp_status ensure_bal_scratch(fp_ctx* ctx, int R) {
  const size_t ntiles = (size_t)(R + TILE - 1) / TILE;
  const size_t need = ntiles * (size_t)ctx->K;
  if (need > ctx->hist_cap) {
    FP_TRY(dalloc(ctx, &ctx->hist, need));
    FP_TRY(dalloc(ctx, &ctx->pref, need));
    fill_async<int>(ctx, ctx->hist, need, 0);
    ctx->hist_cap = need;
  }
  return FP_OK;
}

// The apply's blocks and their nets: about APPLY_NET_BLOCKS blocks, of 16 to
// APPLY_NETS nets each; few nets of more than 64 pins, which a wavefront each
// replays, go one to a wavefront (2,000 nets of 1,500 pins at K = 1024: 58 us
// a round in blocks of 16 nets, 22 in blocks of 4).
int apply_blocks(const fp_ctx* ctx, int& per_block) {
  const int least = ctx->pins > (long long)WAVE * ctx->noe ? APPLY_BLOCK / WAVE : 16;
  per_block = std::max(least, std::min(APPLY_NETS, (ctx->noe + APPLY_NET_BLOCKS - 1) / APPLY_NET_BLOCKS));
  return std::max(1, (ctx->noe + per_block - 1) / per_block);
}

// Whether a sub-round of the stream hands its touched nets to the apply as a list.
// Looking for them among all nets' stamps costs a launch in proportion to the
// nets, and leaves some blocks many of the few touched ones; a list costs the admission
// an exchange a pin and an atomic per 64 slots on one counter. Whole streams,
// K = 64 (16 for the first), stamps and list, ms:
//   slots                 256          1,024        4,096       16,384      32,768
//   1,000,000 Zipf     220  202      72.5 53.2    20.4 15.9    6.3  5.6    3.9  4.0
//   2,000,000 of 13                   372  115    98.9 36.1   29.0 15.8   17.3 12.6
//   600,000 of 9       211  115      67.9 30.6    18.0  9.0    5.3  3.6    3.2  2.8
//   300,000 of 9        86   58      22.3 15.3     6.2  4.5    2.1  1.9    1.4  1.4
//   200,000 Zipf      35.0 37.5       9.4 10.0     2.7  2.9    1.1  1.3
// Passes of the balanced schedule, whose rounds move few vertices, take the stamps:
// 300,000 nets, rounds of 256, 15.8 ms against 17.6; 1,000,000, of 16,384, 2.29 against 2.17.
bool apply_by_list(const fp_ctx* ctx, int nslots) {
  return ctx->noe >= APPLY_LIST_NOE && (long long)nslots * APPLY_LIST_RATIO <= ctx->noe;
}

void launch_apply(fp_ctx* ctx, ApplyArgs& ap, int extra_blocks, bool list) {
  const int K = ctx->K;
  const bool indexed = apply_indexed(K, list);
  ap.noe = ctx->noe;
  ap.net_ptr = ctx->net_ptr;
  ap.apply_pins = ctx->apply_pins;
  ap.slot_own = ctx->slot_own;
  ap.slot_dec = ctx->slot_dec;
  ap.net_stamp = ctx->net_stamp;
  ap.touched = ctx->touched;
  ap.tcount = ctx->counters;
  ap.ent = ctx->ent;
  ap.ev = ctx->ev;
  ap.mask_words = mask_words(K);
  ap.K = K;
  ap.pb = ctx->pb;
  ap.pmask = ctx->pmask;
  ap.net_blocks = apply_blocks(ctx, ap.per_block);
  ap.lane_words = apply_lane_words(K);
  ap.wave_bytes = (int)apply_wave_bytes(K, indexed);
  auto kernel = list ? (indexed ? k_apply<true, true> : k_apply<false, true>)
                     : (indexed ? k_apply<true, false> : k_apply<false, false>);
  kernel<<<ap.net_blocks + extra_blocks, APPLY_BLOCK, apply_lds(K, list), ctx->stream>>>(ap);
}

// the scan and the admission of a BAL round (first_free: of a sub-round of the stream)
void launch_admission(fp_ctx* ctx, int r0, int nslots, int ntiles, long long cap, bool first_free, unsigned tag,
                      bool list) {
  const int K = ctx->K;
  if (ntiles <= SCAN_WAVE_TILES)
    k_bal_scan<true><<<std::max(1, std::min((K + 3) / 4, 1024)), 256, 0, ctx->stream>>>(
        ctx->hist, ctx->pref, ntiles, K, ctx->sizes_frozen, cap, ctx->over, ctx->counters);
  else
    k_bal_scan<false><<<std::max(1, std::min(K, 1024)), 256, 0, ctx->stream>>>(ctx->hist, ctx->pref, ntiles, K,
                                                                               ctx->sizes_frozen, cap, ctx->over,
                                                                               ctx->counters);
  // the size changes are summed per block in LDS where K parts fit, and every
  // block then adds to the K size words, one after another: larger blocks where
  // that still leaves many. us with blocks of 256, 512 and 1,024, K = 16 and 256:
  //   16,384 slots    5.0  5.4  6.4     7.5  8.7 11.3
  //   65,536          8.0  7.8  9.7     8.5  8.7 11.4
  //   131,072        12.6 10.9 12.9    10.7  9.5 11.8
  //   262,144        17.7 13.7 13.5    15.8 12.8 13.0
  const int ablock = ntiles >= 2048 ? ADMIT_BLOCK : 256;
  const int tiles = ablock / WAVE;  // per block
  const int agrid = std::max(1, std::min((ntiles + tiles - 1) / tiles, 4096));
  const size_t lds = (size_t)K * sizeof(long long);
  const bool agg = lds <= (size_t)LDS_BUDGET;
  auto admit = list ? (agg ? k_bal_admit<true, true> : k_bal_admit<false, true>)
                    : (agg ? k_bal_admit<true, false> : k_bal_admit<false, false>);
  admit<<<agrid, ablock, agg ? lds : 0, ctx->stream>>>(
      ctx->slot_dec, ctx->slot_own, ctx->order, ctx->vwgt, r0, nslots, ntiles, K, ctx->sizes_frozen, cap, first_free,
      ctx->over, ctx->pref, ctx->part, ctx->sizes, ctx->moves, ctx->vtx_ptr, ctx->vtx_nets, tag, ctx->net_stamp,
      ctx->touched, ctx->counters);
}

fp_status check_sched(fp_ctx* ctx, const fp_schedule* s) {
  if (!s) return fail(ctx, FP_ERR_ARG, "null schedule");
  if (s->kind != FP_SCHED_REF && s->kind != FP_SCHED_BAL) return fail(ctx, FP_ERR_ARG, "unknown schedule kind %d", s->kind);
  if (s->round < 1) return fail(ctx, FP_ERR_ARG, "round size must be >= 1");
  if (!(s->ldg_C > 0)) return fail(ctx, FP_ERR_ARG, "ldg_C must be > 0");
  return FP_OK;
}

// what the evaluation kernel's packed keys assume
fp_status check_envelope(fp_ctx* ctx) {
  if (eval_waves(ctx->K) == 0) return fail(ctx, FP_ERR_UNSUPPORTED, "K = %d needs more LDS than a workgroup has", ctx->K);
  if ((unsigned long long)ctx->max_vdeg + 1 >= (1ull << (32 - ctx->pb)))
    return fail(ctx, FP_ERR_UNSUPPORTED, "a vertex of degree %u is too large for K = %d", ctx->max_vdeg, ctx->K);
  if (ctx->total_weight >= (1ll << 31)) return fail(ctx, FP_ERR_UNSUPPORTED, "total vertex weight >= 2^31");
  return FP_OK;
}

EvalArgs make_eval_args(fp_ctx* ctx, const fp_schedule* s) {
  EvalArgs a{};
  a.pad_seg = (unsigned)((size_t)ctx->pins + (size_t)ctx->noe);
  a.vtx_ptr = ctx->vtx_ptr;
  a.vtx_nets = ctx->vtx_nets;
  a.vtx_seg = ctx->vtx_seg;
  a.ev = ctx->ev;
  a.part = ctx->part;
  a.order = ctx->order;
  a.vwgt = ctx->vwgt;
  a.sizes = ctx->sizes;
  a.K = ctx->K;
  a.pb = ctx->pb;
  a.pmask = ctx->pmask;
  a.C = s->ldg_C;
  a.max_pw = s->max_pw;
  a.min_pw = s->min_pw;
  a.slot_own = ctx->slot_own;
  a.slot_dec = ctx->slot_dec;
  return a;
}

}  // namespace

long long tv_scratch_bytes(int K, int R, bool bal) {
  return array_bytes(8ll * R, 2) + (bal ? array_bytes(BAL_BYTES * K * ((R + TILE - 1) / TILE), 2) : 0);
}

fp_status plan_tv(fp_ctx* ctx, RefinePlan& p) {
  const int K = ctx->K;
  const int waves = p.eval_waves > 0 ? std::min(p.eval_waves, eval_waves(K)) : eval_waves(K);
  if (waves == 0) return fail(ctx, FP_ERR_UNSUPPORTED, "K = %d needs more LDS than a workgroup has", K);
  p.eval_waves = waves;
  if (apply_lds(K, true) + apply_static(true) > (size_t)LDS_BUDGET) return fail(ctx, FP_ERR_UNSUPPORTED, "K = %d too large for the apply kernel", K);
  p.R = std::min(p.sched.round, ctx->nov);
  FP_TRY(ensure_round_scratch(ctx, p.R));
  if (p.sched.kind == FP_SCHED_BAL) FP_TRY(ensure_bal_scratch(ctx, p.R));
  // the part masks of the resident lists, kept in step by the passes
  p.masks = ensure_masks(ctx);
  if (p.masks) build_masks(ctx, p.masks);
  return FP_OK;
}

fp_status pass_tv(fp_ctx* ctx, const RefinePlan& p) {
  const int nov = ctx->nov, K = ctx->K, R = p.R, waves = p.eval_waves;
  const fp_schedule* sched = &p.sched;
  const bool bal = sched->kind == FP_SCHED_BAL;
  const size_t lds_e = eval_lds(K, waves);
  // every pass restarts its round tags: clear the stamps
  pass_begin(ctx, nullptr, 0, nullptr);
  unsigned tag = 0;
  for (int r0 = 0; r0 < nov; r0 += R) {
    const int nslots = std::min(R, nov - r0);
    const int ntiles = (nslots + TILE - 1) / TILE;
    tag++;
    EvalArgs a = make_eval_args(ctx, sched);
    a.r0 = r0;
    a.nslots = nslots;
    a.ntiles = ntiles;
    a.tag = tag;
    if (!bal) a.net_stamp = ctx->net_stamp;  // BAL: k_bal_admit stamps the admitted moves' nets
    if (bal) {
      a.hist = ctx->hist;
      a.sizes_frozen = ctx->sizes_frozen;
    }
    if (p.masks) {
      a.masks = p.masks;
      a.noe = ctx->noe;
      a.last_pin = mask_last_pin(ctx);
      const int grid = mask_eval_grid(nslots, p.eval_grid, EVAL_BLOCK / WAVE);
      FP_TRY(launch_timed(ctx, eval_masks_kernel<EVAL_REFINE>(K, mask_wide(ctx)), grid, EVAL_BLOCK, 0, a));
    } else {
      int grid = eval_grid(nslots, waves);
      if (p.eval_grid > 0) grid = std::min(grid, p.eval_grid);
      FP_TRY(launch_timed(ctx, k_tv_eval<EVAL_REFINE>, grid, waves * WAVE, lds_e, a));
    }
    if (bal) {
      launch_admission(ctx, r0, nslots, ntiles, sched->cap, false, tag, false);
    }
    ApplyArgs ap{};
    ap.tag = tag;
    ap.masks = p.masks;
    ap.r0 = r0;
    ap.r1 = r0 + nslots;
    if (!bal) {
      ap.order = ctx->order;
      ap.part = ctx->part;
      ap.sizes = ctx->sizes;
      ap.moves = ctx->moves;
    }
    launch_apply(ctx, ap, bal ? 0 : (nslots + APPLY_BLOCK - 1) / APPLY_BLOCK, false);
  }
  return FP_OK;
}

fp_status plan_refine(fp_ctx* ctx, fp_metric metric, const fp_schedule* sched, RefinePlan& p) {
  if (!ctx->has_state) return fail(ctx, FP_ERR_STATE, "refinement before a state was set");
  if (ctx->dup_pins) return fail(ctx, FP_ERR_UNSUPPORTED, "a net lists the same vertex twice; refinement needs distinct pins");
  const int waves = p.eval_waves, grid = p.eval_grid;
  p = RefinePlan{};
  p.metric = metric;
  p.eval_waves = waves;
  p.eval_grid = grid;
  FP_HIP_OK(hipSetDevice(ctx->device));
  if (metric == FP_METRIC_CN) return plan_cn(ctx, p);  // the lambda = 2 push takes no schedule
  FP_TRY(check_sched(ctx, sched));
  p.sched = *sched;
  FP_TRY(check_envelope(ctx));
  switch (metric) {
    case FP_METRIC_TV: return plan_tv(ctx, p);
    case FP_METRIC_MSV:
    case FP_METRIC_MSRV: return plan_vol(ctx, p);
    case FP_METRIC_TM:
    case FP_METRIC_MSM: return plan_conn(ctx, p);
    default: return fail(ctx, FP_ERR_UNSUPPORTED, "refinement for metric %d not available", (int)metric);
  }
}

fp_status record_pass(fp_ctx* ctx, const RefinePlan& p) {
  switch (p.metric) {
    case FP_METRIC_TV: return pass_tv(ctx, p);
    case FP_METRIC_CN: return pass_cn(ctx, p);
    case FP_METRIC_MSV:
    case FP_METRIC_MSRV: return pass_vol(ctx, p);
    default: return pass_conn(ctx, p);
  }
}

}  // namespace fpe

using namespace fpe;

extern "C" {

fp_status fp_refine(fp_ctx* ctx, fp_metric metric, int passes, const fp_schedule* sched, fp_refine_stats* stats) {
  if (!ctx) return FP_ERR_ARG;
  if (passes < 0) return fail(ctx, FP_ERR_ARG, "passes < 0");
  RefinePlan p;
  FP_TRY(plan_refine(ctx, metric, sched, p));
  fill_async<unsigned long long>(ctx, ctx->moves, 1, 0ull);
  ctx->timed_next = 2;
  ctx->timed_launches = 0;
  ctx->timed_ms = 0;
  hipEvent_t e0 = pooled_event(ctx, 0), e1 = pooled_event(ctx, 1);
  if (!e0 || !e1) return fail(ctx, FP_ERR_HIP, "hipEventCreate failed");
  FP_HIP_OK(hipEventRecord(e0, ctx->stream));
  if (metric == FP_METRIC_CN) {
    FP_TRY(cn_passes(ctx, p, passes));
  } else {
    for (int it = 0; it < passes; it++) FP_TRY(record_pass(ctx, p));
  }
  FP_HIP_OK(hipGetLastError());
  FP_HIP_OK(hipEventRecord(e1, ctx->stream));
  unsigned long long mv = 0;
  FP_TRY(d2h(ctx, &mv, ctx->moves, 1));
  FP_HIP_OK(hipStreamSynchronize(ctx->stream));
  float ms = 0;
  FP_HIP_OK(hipEventElapsedTime(&ms, e0, e1));
  for (size_t i = 2; i + 1 < ctx->timed_next; i += 2) {
    float t = 0;
    FP_HIP_OK(hipEventElapsedTime(&t, ctx->ev_pool[i], ctx->ev_pool[i + 1]));
    ctx->timed_ms += t;
    ctx->timed_launches++;
  }
  if (stats) {
    stats->moves = (long long)mv;
    stats->rounds = metric == FP_METRIC_CN ? passes : (long long)passes * ((ctx->nov + p.R - 1) / p.R);
    stats->pin_visits = (long long)passes * ctx->pins;
    stats->device_ms = ms;
  }
  return FP_OK;
}

fp_status fp_initial_partition_device(fp_ctx* ctx, int mode, int K, int round, double C, long long max_pw,
                                      long long cap, fp_init_stats* stats) {
  if (!ctx) return FP_ERR_ARG;
  if (!ctx->has_graph) return fail(ctx, FP_ERR_STATE, "fp_initial_partition_device before fp_upload");
  if (mode < 0 || mode > 2) return fail(ctx, FP_ERR_ARG, "unknown initial partition mode %d", mode);
  if (round < 1) return fail(ctx, FP_ERR_ARG, "round size must be >= 1");
  if (!(C > 0)) return fail(ctx, FP_ERR_ARG, "C must be > 0");
  if (ctx->dup_pins) return fail(ctx, FP_ERR_UNSUPPORTED, "a net lists the same vertex twice");
  FP_HIP_OK(hipSetDevice(ctx->device));
  FP_TRY(ensure_k(ctx, K));
  FP_TRY(check_envelope(ctx));
  if (apply_lds(K, true) + apply_static(true) > (size_t)LDS_BUDGET) return fail(ctx, FP_ERR_UNSUPPORTED, "K = %d too large for the apply kernel", K);
  const int nov = ctx->nov;
  const int R = std::max(1, std::min(round, nov));
  const int waves = eval_waves(K);
  FP_TRY(ensure_round_scratch(ctx, R));
  FP_TRY(ensure_bal_scratch(ctx, R));
  // the empty state: no part, empty lists, zero sizes
  const size_t segs = (size_t)ctx->pins + (size_t)ctx->noe + ENT_PAD;
  fill_async<int>(ctx, ctx->part, (size_t)std::max(nov, 1), -1);
  fill_async<unsigned>(ctx, ctx->ent, segs, 0u);
  fill_async<unsigned short>(ctx, ctx->ev, segs, (unsigned short)0);
  unsigned long long* masks = ensure_masks(ctx);
  if (masks) fill_async<unsigned long long>(ctx, masks, ((size_t)ctx->noe + 1) * (size_t)(2 * mask_words(K)), 0ull);
  fill_async<long long>(ctx, ctx->sizes, (size_t)K, 0);
  fill_async<unsigned long long>(ctx, ctx->moves, 1, 0ull);
  pass_begin(ctx, nullptr, 0, nullptr);
  hipEvent_t e0 = pooled_event(ctx, 0), e1 = pooled_event(ctx, 1);
  if (!e0 || !e1) return fail(ctx, FP_ERR_HIP, "hipEventCreate failed");
  FP_HIP_OK(hipEventRecord(e0, ctx->stream));
  const int eval_mode = mode == 2 ? EVAL_INIT_CN : EVAL_INIT;
  const size_t lds_e = eval_lds(K, waves);
  int* fb = ctx->counters + 2;
  unsigned tag = 0;
  long long subrounds = 0, rounds = 0;
  int burst = 1;  // sub-rounds enqueued before the host looks at the progress
  auto subround = [&](int r0, int nslots) -> fp_status {
    const int ntiles = (nslots + TILE - 1) / TILE;
    tag++;
    EvalArgs a{};
    a.pad_seg = (unsigned)((size_t)ctx->pins + (size_t)ctx->noe);
    a.vtx_ptr = ctx->vtx_ptr;
    a.vtx_nets = ctx->vtx_nets;
    a.vtx_seg = ctx->vtx_seg;
    a.ev = ctx->ev;
    a.part = ctx->part;
    a.order = ctx->order;
    a.vwgt = ctx->vwgt;
    a.sizes = ctx->sizes;
    a.K = K;
    a.pb = ctx->pb;
    a.pmask = ctx->pmask;
    a.C = C;
    a.max_pw = mode == 0 ? max_pw : LLONG_MAX;
    a.min_pw = LLONG_MIN;
    a.slot_own = ctx->slot_own;
    a.slot_dec = ctx->slot_dec;
    a.r0 = r0;
    a.nslots = nslots;
    a.ntiles = ntiles;
    a.tag = tag;
    a.hist = ctx->hist;
    a.sizes_frozen = ctx->sizes_frozen;
    a.fb_out = fb;
    a.masks = masks;
    a.noe = ctx->noe;
    a.last_pin = mask_last_pin(ctx);
    const int grid = masks ? mask_eval_grid(nslots, 0, EVAL_BLOCK / WAVE) : eval_grid(nslots, waves);
    if (masks)
      (eval_mode == EVAL_INIT_CN ? eval_masks_kernel<EVAL_INIT_CN>(K, false)
                                 : eval_masks_kernel<EVAL_INIT>(K, mask_wide(ctx)))<<<grid, EVAL_BLOCK, 0, ctx->stream>>>(a);
    else if (eval_mode == EVAL_INIT_CN)
      k_tv_eval<EVAL_INIT_CN><<<grid, waves * WAVE, lds_e, ctx->stream>>>(a);
    else
      k_tv_eval<EVAL_INIT><<<grid, waves * WAVE, lds_e, ctx->stream>>>(a);
    k_init_fallback<<<1, 1024, 0, ctx->stream>>>(ctx->slot_dec, ctx->order, ctx->vwgt, r0, nslots, ntiles, K, fb,
                                                 ctx->hist);
    const bool list = apply_by_list(ctx, nslots);
    launch_admission(ctx, r0, nslots, ntiles, cap, true, tag, list);
    ApplyArgs ap{};
    ap.tag = tag;
    ap.masks = masks;
    ap.r0 = r0;
    ap.r1 = r0 + nslots;
    launch_apply(ctx, ap, 0, list);
    FP_HIP_OK(hipGetLastError());
    subrounds++;
    return FP_OK;
  };
  for (int r0 = 0; r0 < nov; r0 += R) {
    const int nslots = std::min(R, nov - r0);
    rounds++;
    // every sub-round places at least one vertex of the round: a round takes
    // at most nslots of them
    int launched = 0;
    for (;;) {
      const int n = std::min(burst, nslots - launched);
      for (int i = 0; i < n; i++) FP_TRY(subround(r0, nslots));
      launched += n;
      unsigned long long placed = 0;
      FP_TRY(d2h(ctx, &placed, ctx->moves, 1));
      FP_HIP_OK(hipStreamSynchronize(ctx->stream));
      if (placed == (unsigned long long)r0 + (unsigned long long)nslots) break;
      if (launched >= nslots)
        return fail(ctx, FP_ERR_STATE, "initial partition round at %d did not place its vertices", r0);
    }
    // the next round starts with as many sub-rounds as this one took (one
    // fewer when this one was done at its first look, to probe downwards)
    burst = launched == burst ? std::max(1, burst - 1) : launched;
  }
  FP_HIP_OK(hipEventRecord(e1, ctx->stream));
  FP_HIP_OK(hipStreamSynchronize(ctx->stream));
  ctx->has_state = true;
  if (stats) {
    float ms = 0;
    FP_HIP_OK(hipEventElapsedTime(&ms, e0, e1));
    stats->rounds = rounds;
    stats->subrounds = subrounds;
    stats->device_ms = ms;
  }
  return FP_OK;
}

fp_status fp_eval_moves(fp_ctx* ctx, fp_metric metric, const fp_schedule* sched, int* dec, int* gain) {
  if (!ctx) return FP_ERR_ARG;
  if (!ctx->has_state) return fail(ctx, FP_ERR_STATE, "fp_eval_moves before a state was set");
  FP_TRY(check_sched(ctx, sched));
  if (metric != FP_METRIC_TV) return fail(ctx, FP_ERR_UNSUPPORTED, "move evaluation for metric %d not available", (int)metric);
  const int nov = ctx->nov, K = ctx->K;
  FP_TRY(check_envelope(ctx));
  const int waves = eval_waves(K);
  FP_HIP_OK(hipSetDevice(ctx->device));
  FP_TRY(ensure_round_scratch(ctx, nov));
  int *d_dec = nullptr, *d_gain = nullptr;
  FP_HIP_OK(hipMalloc(&d_dec, sizeof(int) * (size_t)nov));
  if (hipMalloc(&d_gain, sizeof(int) * (size_t)nov) != hipSuccess) {
    (void)hipFree(d_dec);
    return fail(ctx, FP_ERR_OOM, "hipMalloc failed");
  }
  EvalArgs a = make_eval_args(ctx, sched);
  a.r0 = 0;
  a.nslots = nov;
  a.ntiles = (nov + TILE - 1) / TILE;
  a.dec_out = d_dec;
  a.gain_out = d_gain;
  k_tv_eval<EVAL_REFINE><<<eval_grid(nov, waves), waves * WAVE, eval_lds(K, waves), ctx->stream>>>(a);
  fp_status st = FP_OK;
  if (hipGetLastError() != hipSuccess) st = fail(ctx, FP_ERR_HIP, "k_tv_eval launch failed");
  if (st == FP_OK && dec) st = d2h(ctx, dec, d_dec, (size_t)nov);
  if (st == FP_OK && gain) st = d2h(ctx, gain, d_gain, (size_t)nov);
  if (hipStreamSynchronize(ctx->stream) != hipSuccess && st == FP_OK) st = fail(ctx, FP_ERR_HIP, "sync failed");
  (void)hipFree(d_dec);
  (void)hipFree(d_gain);
  return st;
}

}  // extern "C"
