// modwt.hip -- host side of the level-fused MODWT: level-group planning and
// launches.  The kernels and their design notes are in modwt_kern.h; they
// are instantiated per (element type, filter) in modwt_<type>_<filter>.hip.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "modwt_kern.h"
#include "modwt_tile.h"
#include "wh_common.h"
#include "wh_internal.h"

namespace wh {

namespace {

static_assert(tile_r(false) <= 8 && tile_r(true) <= 8, "a tile group may start at level 3");
constexpr int kNT1 = 512;   // threads, group starting at level 1 (R = 1)
constexpr int kNTR = 256;   // threads, deeper groups (R = 32)
constexpr int kRdeep = 32;
// segments per CU of the deeper groups: their chunks are small (M = 16
// positions of 32 residues), so several workgroups per CU keep enough
// loads in flight (measured at LA8, J = 10, n = 2^24: inverse 0.532 ms with
// one, 0.498 ms with four)
constexpr int kDeepSegPerCu = 4;

struct Group {
  bool tile = false;  // one tile per workgroup (modwt_tile.h) instead of a sliding window
  bool wide = false;  // all levels in one wide tile
  int j0, g, R, NT, M;
  int64_t P;
  int nseg, warm, nchunks;
  size_t lds;
};

// Planner choices the tuner may change (defaults: the rules below).
struct PlanKnobs {
  int g1max = kGmax;                 // deepest first group
  int first_per_cu = 1;              // segments per CU of the first group
  int deep_per_cu = kDeepSegPerCu;   // segments per CU of deeper groups
  int first_nt = kNT1;               // threads of the first inverse group (512, or 256:
                                     // two workgroups per CU in half the LDS); negative: a
                                     // plan of tiles of that many threads, at most g1max
                                     // levels each (g1max 7 or 8: one wide tile)
  bool operator<(const PlanKnobs& o) const {
    return std::tie(g1max, first_per_cu, deep_per_cu, first_nt) <
           std::tie(o.g1max, o.first_per_cu, o.deep_per_cu, o.first_nt);
  }
};

using KnobKey = std::tuple<int, int64_t, int, int, int>;  // inverse, n, J, filter, element size
std::mutex g_knob_mu;
std::map<KnobKey, PlanKnobs> g_knobs;

// whether a launch's shape can be one wide tile: whole tiles of `per`
// positions, FP32, 3..8 levels
bool wide_fits(int per, int64_t n, int J, size_t esz) {
  return esz == 4 && J >= kWideGmin && J <= kWideGmax && n >= per;
}

std::vector<Group> plan_groups(bool inverse, int64_t n, int J, int L, size_t esz,
                               const PlanKnobs& k, int64_t count = 1);
std::vector<Group> plan_tiles(bool inverse, int64_t n, int J, int L, size_t esz,
                              const PlanKnobs& k);

// elements of a tile launch, the padding of sequences that are shorter than a
// tile among them
int64_t padded_elems(const Group& G, int64_t count) {
  return (int64_t(1) << G.j0) * G.nseg * G.M * count;
}

// Default plan knobs, measured on MI355X (replayed graphs, three sets of
// buffers in turn; us, sliding windows -> tiles, LA8 / Haar):
//  * the inverse of a launch of up to 2^21 samples (length times signals)
//    runs as tiles: n = 2^14, J = 8 FP64 21.0 -> 9.0 / 18.6 -> 7.2; 2^18,
//    J = 10 36.4 -> 14.2 / 34.2 -> 11.3; 2^20, J = 10 57.2 -> 36.5 /
//    41.0 -> 30.7; 2^21, J = 10 77.7 -> 66.5 / 64.3 -> 56.1 (FP32 49.0 ->
//    46.0 / 36.1 -> 35.4); at 2^22 the two are level in FP64 and the sliding
//    windows ahead in FP32 (82.6 against 87.7).  Tiles of 256 threads up to
//    2^17 samples (2^17, J = 9: 10.8 against 11.5), 512 beyond (2^18, J = 10:
//    14.2 against 15.7);
//  * not where a deeper group's sequences, n / 2^j0 long, leave most of a tile
//    empty and the sliding windows need only one or two groups (Haar, calls back
//    to back: 1024 x 2^8, J = 8 FP32, padding 16 to 1, 17.5 against 21.4; 256 x
//    2^12, J = 12 FP64, 16 to 1, 55.5 against 84; 256 x 2^13, J = 12, 2^24 elements
//    padded 8 to 1, 88 against 105; but 1024 x 2^10, J = 10 FP64, 8 to 1, 87.9 -> 52.6;
//    64 x 2^12, J = 12, 16 to 1, five sliding groups, 34.4 -> 26.6);
//  * the forward of up to 2^18 samples as tiles of 512 threads (2^14, J = 8:
//    18.4 -> 8.9 / 15.8 -> 7.0; 2^18, J = 10: 29.6 -> 16.5 / 26.5 -> 12.9)
//    unless the sliding windows take fewer steps than two chunks a tile group:
//    short signals whose levels all fit one group (n = 2^10, J = 7..10: Haar, two
//    chunks, 4.9 against 6.8 and at 256 signals 7.5 against 10.4; LA8 J = 8, three
//    chunks, 9.2 -> 7.8 and 10.4 -> 9.1);
//  * of up to 2^19 where they take at least three (2^19, J = 10 FP32: 22.7 ->
//    16.2; J = 8 level to 1.1 times ahead; 64 x 2^13, J = 12 Haar FP32, five for
//    three tile groups, 17.0 against 20.3).  Beyond, it is bound by its stores,
//    which the sliding windows make in longer runs (2^20, J = 8 FP32: 18.5 against
//    19.7);
//  * an FP32 inverse of at most 8 levels as one wide tile: with 7 or 8
//    levels, which take two tile groups, from 2^19 samples (64 x 2^13, J = 8
//    LA8 / Haar: 19.2 -> 14.9 / 16.4 -> 11.5; 32 x 2^14 level at 15.3) up to
//    2^23 (512 x 2^14: sliding 152 -> 118 / 111 -> 64; one 2^24 signal 191
//    against 195); with fewer, beyond the tiles' range and below 2^23 (2^22,
//    J = 6 LA8 43.6 -> 39.3, J = 4 31.8 -> 28.9; 512 x 2^14, J = 6 75
//    against 81);
//  * sliding inverses: of up to 2^18 samples a 256-thread first group of at most
//    six levels, two segments per CU (one 512-thread workgroup per CU has too few:
//    2^16 28 -> 25); of one FP32 signal beyond 2^20 the same with four (half the
//    FP64 LDS, so several workgroups share a CU): n = 2^22 90 -> 83, 2^24 307 -> 258.
// Rules for the FP64 sliding windows taken from the tuner's isolated
// timings were slower in the pipeline (what the other transform leaves in
// the last-level cache matters as much as the plan), so those keep the plain
// defaults.
PlanKnobs default_knobs(bool inverse, int64_t n, int64_t count, int J, int filt, size_t esz) {
  const int64_t total = n * count;
  const int L = filter_length(filt);
  const bool deep = J > kTileGmax;  // two tile groups or more
  PlanKnobs k;
  if (inverse && wide_fits(kWideInvP, n, J, esz) &&
      (deep ? total >= (int64_t(1) << 19) && total <= (int64_t(1) << 23)
            : total > (int64_t(1) << 21) && total < (int64_t(1) << 23))) {
    k.first_nt = -kWideInvNT;
    k.g1max = kWideGmax;
    return k;
  }
  if (inverse && (total <= (int64_t(1) << 18) ||
                  (count == 1 && esz == 4 && n > (int64_t(1) << 20)))) {
    k.first_nt = kNT1 / 2;
    k.first_per_cu = total <= (int64_t(1) << 18) ? 2 : 4;
    k.g1max = 6;
  }
  if (total > (int64_t(1) << (inverse ? 21 : 19))) return k;
  PlanKnobs t;
  t.first_nt = inverse && total <= (int64_t(1) << 17) ? -kNT1 / 2 : -kNT1;
  t.g1max = kTileGmax;
  if (!deep && (inverse || total <= (int64_t(1) << 18))) return t;
  const auto sliding = plan_groups(inverse, n, J, L, esz, k, count);
  if (!deep) return sliding.size() > 1 ? t : k;
  const auto tiles = plan_tiles(inverse, n, J, L, esz, t);
  if (inverse) {
    int64_t padded = 0;
    for (const Group& G : tiles) padded = std::max(padded, padded_elems(G, count));
    const bool full = padded <= 8 * total && padded <= (int64_t(1) << 23);
    return full || sliding.size() > 2 ? t : k;
  }
  size_t chunks = 0;
  for (const Group& G : sliding) chunks += size_t(G.nchunks);
  const bool pays = total <= (int64_t(1) << 18) ? chunks > tiles.size() : chunks >= 3 * tiles.size();
  return pays ? t : k;
}

PlanKnobs knobs_for(bool inverse, int64_t n, int J, int filt, size_t esz, int64_t count = 1) {
  std::lock_guard<std::mutex> lk(g_knob_mu);
  auto it = g_knobs.find(KnobKey{inverse ? 1 : 0, n, J, filt, int(esz)});
  // tuned on one signal: tiles chosen there say nothing about a larger launch
  const bool use = it != g_knobs.end() && (count == 1 || it->second.first_nt > 0);
  return use ? it->second : default_knobs(inverse, n, count, J, filt, esz);
}

// Tile groups: levels 1..J in ceil(J / depth) groups of nearly equal depth.
// A first of several groups has at least three levels, so that the next one's
// 2^{j0} residues make whole blocks of tile_r.
std::vector<Group> plan_tiles(bool inverse, int64_t n, int J, int L, size_t esz,
                              const PlanKnobs& k) {
  std::vector<Group> gs;
  const int NT = -k.first_nt;
  if (k.g1max > kTileGmax) {
    Group G{};
    G.tile = G.wide = true;
    G.g = J;
    G.R = 1;
    G.NT = NT;
    G.P = inverse ? kWideInvP : kWideGradP;
    G.M = int(G.P);
    G.nseg = int(n / G.P);
    G.warm = tile_halo(L, J);
    G.nchunks = 1;
    G.lds = size_t(G.P + G.warm) * (inverse ? 2 : 1) * esz;
    gs.push_back(G);
    return gs;
  }
  const int cap = std::min(k.g1max, kTileGmax);
  const int deep = std::min(cap, kTileGmax - 1);
  const int ng = J <= cap ? 1 : (J + deep - 1) / deep;
  int j0 = 0;
  for (int i = 0; i < ng; ++i) {
    Group G{};
    G.tile = true;
    G.j0 = j0;
    G.g = (J - j0 + (ng - i) - 1) / (ng - i);
    if (i == 0 && ng > 1) G.g = std::max(G.g, 3);
    G.R = j0 == 0 ? 1 : tile_r(inverse);
    G.NT = NT;
    G.M = 2 * NT / G.R;
    G.P = G.M;
    G.nseg = int(std::max<int64_t>(1, (n >> j0) / G.P));
    G.warm = tile_halo(L, G.g);
    G.nchunks = 1;
    const size_t top = size_t(2 * NT + tile_halo(L, G.g) * G.R);
    const size_t below = size_t(2 * NT + tile_halo(L, G.g - 1) * G.R);
    G.lds = inverse ? 2 * (top + (G.g > 1 ? below : 0)) * esz
                    : (top + size_t(2 * NT + (G.warm - tile_halo(L, 1)) * G.R)) * esz;
    gs.push_back(G);
    j0 += G.g;
  }
  return gs;
}

// LDS elements of one residue's buffers (the first inverse group keeps the
// linear buffers of InvLinCtx, deeper inverse groups rings)
size_t ring_elems(bool inverse, int L, int g, int M, int R) {
  if (!inverse) return size_t(fwd_off(L, M, g));
  return size_t(2) * (R == 1 ? lin_off(L, M, g + 1) : inv_off(L, M, g + 1));
}

int64_t round_up64(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

// Partition levels 1..J into groups.  The first group (R = 1) fuses at
// least min(J, 5) levels, so deeper groups start at a stride of 32 or more
// and run R = 32 residues; every group fuses as many levels as the LDS
// budget allows while its warm-up stays at most half a segment (one
// segment per CU for the first group, kDeepSegPerCu for deeper ones).
std::vector<Group> plan_groups(bool inverse, int64_t n, int J, int L, size_t esz,
                               const PlanKnobs& k, int64_t count) {
  if (k.first_nt < 0) return plan_tiles(inverse, n, J, L, esz, k);
  const DeviceInfo& dev = device_info();
  const size_t budget = std::min<size_t>(dev.max_lds_per_block, 160 * 1024) - 1024;
  const int64_t cus = std::max(1, dev.num_cus);
  std::vector<Group> gs;
  int j0 = 0;
  while (j0 < J) {
    Group G{};
    G.j0 = j0;
    const int64_t B = int64_t(1) << j0;
    G.R = (j0 == 0) ? 1 : kRdeep;
    G.NT = (G.R == 1) ? (inverse ? k.first_nt : kNT1) : kNTR;
    // a 256-thread first inverse group plans for two workgroups per CU
    const size_t gbudget = (G.R == 1 && G.NT < kNT1) ? budget / 2 : budget;
    const int64_t Nm = n >> j0;
    G.M = int(std::min<int64_t>(2 * G.NT / G.R, Nm));
    const int64_t nrb = B / G.R;
    // segments per signal: the CUs' worth of workgroups is shared by the
    // `count` signals of a many-signal launch
    const int64_t target = std::max<int64_t>(
        1, (j0 == 0 ? k.first_per_cu : k.deep_per_cu) * cus / (nrb * std::max<int64_t>(1, count)));
    int64_t nseg_t = 1;
    while (nseg_t * 2 <= target && Nm / (nseg_t * 2) >= G.M) nseg_t *= 2;
    const int64_t Pt = Nm / nseg_t;
    const int gmin = (j0 == 0) ? std::min(J, 5) : 1;
    int gbest = gmin;
    const int gcap = (j0 == 0) ? std::max(gmin, std::min(k.g1max, kGmax)) : kGmax;
    for (int g = gmin + 1; g <= std::min(J - j0, gcap); ++g) {
      if (ring_elems(inverse, L, g, G.M, G.R) * G.R * esz > gbudget) break;
      // the first inverse group keeps linear buffers whose windows move once
      // per chunk: a window longer than the chunk would cost more to move
      // than the chunk itself
      if (inverse && G.R == 1 && inv_win(L, g) > G.M) break;
      // the linear buffers' pair mapping takes outputs q and q + s of a
      // chunk, so the group's deepest stride 2^{g-1} must fit twice
      if (inverse && G.R == 1 && (int64_t(1) << g) > G.M) break;
      int64_t warm = round_up64(int64_t(L - 1) * ((int64_t(1) << g) - 1), G.M);
      if (warm > Pt / 2 && nseg_t > 1) break;
      gbest = g;
    }
    G.g = gbest;
    G.warm = int(round_up64(int64_t(L - 1) * ((int64_t(1) << G.g) - 1), G.M));
    int64_t nseg = 1;
    while (nseg * 2 <= target && Nm / (nseg * 2) >= G.M &&
           Nm / (nseg * 2) >= 2 * int64_t(G.warm))
      nseg *= 2;
    G.nseg = int(nseg);
    G.P = Nm / nseg;
    G.nchunks = int((G.P + G.warm) / G.M);
    G.lds = ring_elems(inverse, L, G.g, G.M, G.R) * G.R * esz;
    gs.push_back(G);
    j0 += G.g;
  }
  return gs;
}

// the groups as text: what wh_debug_modwt_plan returns, and what tells one plan
// from another (the kind of a launch among it: a tile and a sliding window may
// agree in depth, segments and threads)
std::string plan_text(const std::vector<Group>& gs) {
  std::string s;
  for (const Group& G : gs) {
    char buf[256];
    snprintf(buf, sizeof buf,
             "{j0=%d g=%d R=%d NT=%d M=%d nseg=%d P=%lld warm=%d chunks=%d lds=%zu%s} ", G.j0,
             G.g, G.R, G.NT, G.M, G.nseg, (long long)G.P, G.warm, G.nchunks, G.lds,
             G.tile ? " tile" : "");
    s += buf;
  }
  return s;
}

template <typename T>
int launch(bool inverse, int filt, const Group& G, const ModwtArgs& a, int64_t count, int sp,
           hipStream_t st, int cand = 1) {
  GroupLaunch gl;
  gl.R = G.R;
  gl.NT = G.NT;
  gl.G = G.g;
  gl.wide = G.wide;
  gl.sp = sp;
  gl.count = count;
  gl.cand = unsigned(cand);
  gl.blocks = ((int64_t(1) << G.j0) / G.R) * G.nseg;
  gl.lds = G.lds;
  if (count < 1 || count > 65535) return set_error(WH_ERR_ARG, "modwt: signal count out of range");
  // element mapping of the R = 1 group: adjacent pairs for the forward
  // (16-byte LDS and HBM accesses; it is write-bound), two outputs of one
  // residue class for the inverse (L + 1 interleaved (S, D) reads instead of
  // 2L; it is LDS-bound)
  gl.map = inverse ? 2 : 0;
  if (G.tile)
    return modwt_tile_launch<T>(inverse ? TileOp::kInverse
                                : sp == kStoreSmooth ? TileOp::kForwardDetails
                                                     : TileOp::kForward,
                                filt, gl, a, GradArgs{}, st);
  if (gl.blocks > 0x7fffffff) return set_error(WH_ERR_ARG, "modwt: grid too large");
  if (inverse && G.R == 1 && (int64_t(1) << G.g) > G.M)
    return set_error(WH_ERR_UNSUPPORTED, "modwt: inverse group deeper than its chunk allows");
  switch (filt) {
    case kHAAR: return modwt_launch<T, kHAAR>(inverse, gl, a, st);
    case kD4: return modwt_launch<T, kD4>(inverse, gl, a, st);
    case kC6: return modwt_launch<T, kC6>(inverse, gl, a, st);
    default: return modwt_launch<T, kLA8>(inverse, gl, a, st);
  }
}

ModwtArgs args_of(const Group& G, int64_t n) {
  ModwtArgs a{};
  a.n = n;
  a.P = G.P;
  a.j0 = G.j0;
  a.g = G.g;
  a.M = G.M;
  a.warm = G.warm;
  a.nchunks = G.nchunks;
  return a;
}

// zeros into S slots (blockIdx.z) of every signal's coefficients (blockIdx.y)
constexpr int kMaxSlots = 64;
struct Slots {
  unsigned char level[kMaxSlots];  // 1-based
};
template <typename T>
__global__ void zero_slots_k(T* __restrict__ p, int64_t n, int64_t per, Slots s) {
  T* q = p + int64_t(blockIdx.y) * per + 2 * n * int64_t(s.level[blockIdx.z] - 1);
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x)
    q[i] = T(0);
}

// the S slots at the groups' boundaries, which carried the next group's input: the
// adjoint of the inverse is zero there
template <typename T>
int zero_handoffs(void* xmod, const std::vector<Group>& groups, int64_t n, int64_t count,
                  int64_t per, hipStream_t st) {
  if (groups.size() < 2) return WH_OK;
  if (groups.size() > kMaxSlots) return set_error(WH_ERR_UNSUPPORTED, "adjoint: too many level groups");
  Slots s{};
  for (size_t gi = 0; gi + 1 < groups.size(); ++gi)
    s.level[gi] = static_cast<unsigned char>(groups[gi].j0 + groups[gi].g);
  const dim3 grid(unsigned(std::min<int64_t>((n + 255) / 256, 1024)), unsigned(count),
                  unsigned(groups.size() - 1));
  hipLaunchKernelGGL(zero_slots_k<T>, grid, dim3(256), 0, st, static_cast<T*>(xmod), n, per, s);
  WH_HIP_CHECK(hipGetLastError());
  return WH_OK;
}

// the tuner's test signal: values uniform in [-1, 1) from a hash of the
// index (a zero signal runs at other speeds than real data does)
template <typename T>
__global__ void tune_signal_k(T* __restrict__ p, int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    uint64_t h = uint64_t(i) * 0x9e3779b97f4a7c15ull;
    h ^= h >> 29;
    h *= 0xbf58476d1ce4e5b9ull;
    h ^= h >> 32;
    p[i] = T(double(h >> 11) * 0x1.0p-52 - 1.0);
  }
}

template <typename T>
int modwt_fwd_t(const void* x, void* xmod, int64_t n, int64_t count, int J, int filt, int sp,
                hipStream_t st) {
  const int L = filter_length(filt);
  PlanKnobs k = knobs_for(false, n, J, filt, sizeof(T), count);
  if (sp == kStoreAdjoint && k.first_nt < 0) k = PlanKnobs{};  // the tiles store a forward only
  auto groups = plan_groups(false, n, J, L, sizeof(T), k, count);
  const int64_t per = 2 * n * J;
  for (const Group& G : groups) {
    ModwtArgs a = args_of(G, n);
    a.in = (G.j0 == 0) ? x : static_cast<const T*>(xmod) + 2 * n * int64_t(G.j0 - 1);
    a.bs_in = (G.j0 == 0) ? n : per;
    a.xmod = xmod;
    a.bs_xmod = per;
    int rc = launch<T>(false, filt, G, a, count, sp, st);
    if (rc) return rc;
  }
  if (sp == kStoreAdjoint) return zero_handoffs<T>(xmod, groups, n, count, per, st);
  return WH_OK;
}

template <typename T>
int modwt_inv_t(const void* xmod, void* x, int64_t n, int64_t count, int J, int filt,
                const wh_thresh* thr, hipStream_t st, void* ws = nullptr, size_t ws_bytes = 0,
                const Candidates& c = Candidates{}) {
  const int L = filter_length(filt);
  const int64_t total = count * c.count;  // signals inverted
  auto groups = plan_groups(true, n, J, L, sizeof(T), knobs_for(true, n, J, filt, sizeof(T), total),
                            total);
  const int64_t per = 2 * n * J;
  // the S_{j0} handed between groups lives in library scratch, or in the
  // caller's workspace `ws` (2 n values per signal: two halves used
  // alternately; every group writes all of its half before the next group
  // reads it, so nothing needs clearing)
  T* scratch = nullptr;
  if (groups.size() > 1) {
    const size_t need = 2 * size_t(n) * size_t(total) * sizeof(T);
    void* p = ws;
    if (ws) {
      if (need > ws_bytes) return set_error(WH_ERR_ARG, "modwt inverse: workspace too small");
    } else {
      int rc = scratch_get(need, &p);
      if (rc) return rc;
    }
    scratch = static_cast<T*>(p);
  }
  const T* stop = static_cast<const T*>(xmod) + 2 * n * int64_t(J - 1);
  int64_t bs_stop = per, bs_stop_z = 0;
  for (int gi = int(groups.size()) - 1; gi >= 0; --gi) {
    const Group& G = groups[gi];
    ModwtArgs a = args_of(G, n);
    a.xmod = const_cast<void*>(xmod);
    a.bs_xmod = per;
    a.stop = stop;
    a.bs_stop = bs_stop;
    T* dst = (G.j0 == 0) ? static_cast<T*>(x) : scratch + (gi & 1) * n * total;
    a.out = dst;
    a.bs_out = n;
    a.bs_out_z = n * count;
    a.bs_stop_z = bs_stop_z;
    if (thr && thr->enabled) {
      a.th_on = 1;
      a.hardness = thr->hardness;
      a.minlevel = thr->minlevel;
      a.maxlevel = thr->maxlevel;
      a.th_value = thr->value;
      a.th_levels = thr->levels;
    }
    int rc = launch<T>(true, filt, G, a, count, kStoreAll, st, c.count);
    if (rc) return rc;
    stop = dst;
    bs_stop = n;
    bs_stop_z = n * count;
  }
  return WH_OK;
}

// The tiles of the adjoint (of the details) and gradient kernels.  FP32
// launches of at most 8 levels run as one wide tile: with 7 or 8 levels from
// 2^19 samples (64 x 2^13, J = 8, LA8: adjoint 19.8 -> 14.0 us, gradient 24.0
// -> 21.6; 512 x 2^14 140 -> 98 and 160 -> 105), with fewer the adjoint
// beyond 2^21 (2^21, J = 6: 21.7 against 24.3; 512 x 2^14, J = 5 D4: 50 ->
// 46) and the gradient from 2^20 (256 x 2^12, J = 6: 22.6 -> 18.5; 2^19: 15.5
// against 17.4).
std::vector<Group> adjoint_tiles(bool inverse, int64_t n, int64_t count, int J, int L,
                                 size_t esz, bool can_wide) {
  PlanKnobs k;
  const int64_t total = n * count;
  const int64_t from = J > kTileGmax ? int64_t(1) << 19
                       : inverse     ? (int64_t(1) << 21) + 1
                                     : int64_t(1) << 20;
  const bool wide =
      can_wide && wide_fits(inverse ? kWideInvP : kWideGradP, n, J, esz) && total >= from;
  k.g1max = wide ? kWideGmax : kTileGmax;
  k.first_nt = wide ? -kWideInvNT : -kTileAdjNT;
  return plan_tiles(inverse, n, J, L, esz, k);
}

GroupLaunch launch_of(const Group& G, int64_t count) {
  GroupLaunch gl{};
  gl.R = G.R;
  gl.NT = G.NT;
  gl.G = G.g;
  gl.wide = G.wide;
  gl.count = count;
  gl.blocks = ((int64_t(1) << G.j0) / G.R) * G.nseg;
  return gl;
}

// One level of the forward's adjoint: out = Sb_{j-1} + H_j^T u + G_j^T Db_j, a
// tap k 2^{j-1} positions back (the terms and order of adjoint1).  Every tap is a
// shifted contiguous read.  Levels whose sequences are too short for tiles.
template <typename T, int FILT>
__global__ __launch_bounds__(256) void fwd_adj_level_k(const T* __restrict__ u0, int64_t bs_u,
                                                       const T* __restrict__ gxm0, int64_t per,
                                                       int j, int with_s, T* __restrict__ out0,
                                                       int64_t n) {
  constexpr int L = Filter<FILT>::L;
  const int64_t sig = blockIdx.y;
  const T* __restrict__ u = u0 + sig * bs_u;
  const T* __restrict__ db = gxm0 + sig * per + 2 * n * int64_t(j - 1) + n;
  const T* __restrict__ sb =
      with_s && j >= 2 ? gxm0 + sig * per + 2 * n * int64_t(j - 2) : nullptr;
  T* __restrict__ out = out0 + sig * n;
  const int64_t s = int64_t(1) << (j - 1), mask = n - 1;
  for (int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x; p < n; p += int64_t(gridDim.x) * 256) {
    T acc = sb ? sb[p] : T(0);
#pragma unroll
    for (int k = 0; k < L; ++k) {
      const int64_t q = (p - k * s) & mask;
      acc = fma(u[q], T(Filter<FILT>::c(k)), acc);
      acc = fma(db[q], T(gcoef<FILT>(k)), acc);
    }
    out[p] = acc;
  }
}

template <typename T>
int fwd_adj_level(const T* u, int64_t bs_u, const T* gxm, int64_t per, int j, bool with_s, T* out,
                  int64_t n, int64_t count, int filt, hipStream_t st) {
  const dim3 grid(unsigned(std::min<int64_t>((n + 255) / 256, 2048)), unsigned(count));
  auto kern = filt == kHAAR ? fwd_adj_level_k<T, kHAAR>
              : filt == kD4 ? fwd_adj_level_k<T, kD4>
              : filt == kC6 ? fwd_adj_level_k<T, kC6>
                            : fwd_adj_level_k<T, kLA8>;
  hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, u, bs_u, gxm, per, j, with_s ? 1 : 0, out, n);
  WH_HIP_CHECK(hipGetLastError());
  return WH_OK;
}

// Whether a group of the forward's adjoint runs level by level: its sequences
// fill an eighth of a tile or less and the launch is large (Haar, whole call, us,
// tiles -> levels: 1024 x 2^12, J = 12 FP64 585 -> 252; 256 x 2^12, J = 12 122 -> 60;
// 1024 x 2^8, J = 8 33.5 -> 20.5; 1024 x 2^10, J = 10 FP32 56 -> 34; short of the line,
// 64 x 2^13, J = 12 FP64, 44 as tiles against 55 with every level a launch).
bool by_level(const Group& G, int64_t n, int64_t count) {
  const int64_t padded = padded_elems(G, count), total = n * count;
  return !G.wide && ((padded >= 16 * total && padded >= (int64_t(1) << 22)) ||
                     (padded >= 8 * total && padded >= (int64_t(1) << 23)));
}

// adjoint of the forward: the level groups from the deepest up
template <typename T>
int fwd_adj_t(const void* gxmod, void* gx, int64_t n, int64_t count, int J, int filt,
              bool details, hipStream_t st) {
  auto groups = adjoint_tiles(true, n, count, J, filter_length(filt), sizeof(T), details);
  const int64_t per = 2 * n * J;
  const T* gxm = static_cast<const T*>(gxmod);
  T* scratch = nullptr;
  if (groups.size() > 1) {
    void* p = nullptr;
    int rc = scratch_get(2 * size_t(n) * size_t(count) * sizeof(T), &p);
    if (rc) return rc;
    scratch = static_cast<T*>(p);
  }
  const T* stop = gxm + 2 * n * int64_t(J - 1);
  int64_t bs_stop = per;
  int half = 0;  // of the scratch, to be written next; the other holds stop
  auto next = [&](bool last) {
    T* dst = last ? static_cast<T*>(gx) : scratch + half * n * count;
    half ^= 1;
    return dst;
  };
  for (int gi = int(groups.size()) - 1; gi >= 0; --gi) {
    const Group& G = groups[gi];
    if (gi > 0 && by_level(G, n, count)) {
      for (int j = G.j0 + G.g; j > G.j0; --j) {
        T* dst = next(false);
        int rc = fwd_adj_level<T>(stop, bs_stop, gxm, per, j, !details, dst, n, count, filt, st);
        if (rc) return rc;
        stop = dst;
        bs_stop = n;
      }
      continue;
    }
    ModwtArgs a = args_of(G, n);
    a.xmod = const_cast<void*>(gxmod);
    a.bs_xmod = per;
    a.stop = stop;
    a.bs_stop = bs_stop;
    T* dst = next(G.j0 == 0);
    a.out = dst;
    a.bs_out = n;
    int rc = modwt_tile_launch<T>(details ? TileOp::kAdjDetails : TileOp::kAdjFull, filt,
                                  launch_of(G, count), a, GradArgs{}, st);
    if (rc) return rc;
    stop = dst;
    bs_stop = n;
  }
  return WH_OK;
}

// workgroups per signal of the groups (partial sums of their levels)
struct GradSums {
  int ngroups;
  int end[8];     // first level beyond the group
  int64_t blocks[8];
};

// glam[l] = the sum of level l's partials over signals and workgroups, in a
// fixed order; zero outside [minlevel, maxlevel]
__global__ __launch_bounds__(256) void grad_sum_k(const double* __restrict__ partial,
                                                  double* __restrict__ glam, int64_t count,
                                                  int64_t per_signal, GradSums gs, int minlevel,
                                                  int maxlevel) {
  const int l = blockIdx.x;
  __shared__ double red[256];
  double acc = 0.0;
  if (l >= minlevel && l <= maxlevel) {
    int g = 0;
    while (l >= gs.end[g]) ++g;
    const int64_t nb = gs.blocks[g];
    const double* p = partial + l * count * per_signal;
    for (int64_t i = threadIdx.x; i < count * nb; i += 256) acc += p[(i / nb) * per_signal + i % nb];
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (int(threadIdx.x) < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) glam[l] = red[0];
}

// adjoint of the thresholding inverse (thr null: of the plain inverse) over
// the coefficients c
template <typename T>
int inv_grad_t(const void* gy, const void* c, void* gc, bool zero_s, double* glam, int64_t n,
               int64_t count, int J, int filt, const wh_thresh* thr, hipStream_t st) {
  auto groups = adjoint_tiles(false, n, count, J, filter_length(filt), sizeof(T), true);
  if (groups.size() > 8) return set_error(WH_ERR_UNSUPPORTED, "adjoint: too many level groups");
  GradArgs q{};
  q.gc = gc;
  q.zero_s = zero_s;
  q.minlevel = 1;  // none
  if (thr) {
    q.hardness = thr->hardness;
    q.minlevel = thr->minlevel;
    q.maxlevel = thr->maxlevel;
    q.value = thr->value;
    q.levels = thr->levels;
  }
  GradSums gs{};
  for (const Group& G : groups) {
    gs.end[gs.ngroups] = G.j0 + G.g;
    gs.blocks[gs.ngroups] = launch_of(G, count).blocks;
    q.per_signal = std::max(q.per_signal, gs.blocks[gs.ngroups]);
    ++gs.ngroups;
  }
  void* p = nullptr;
  if (glam) {
    int rc = stats_get(size_t(J) * size_t(count) * size_t(q.per_signal) * sizeof(double), &p);
    if (rc) return rc;
    q.partial = static_cast<double*>(p);
  }
  // The S between groups: through the cotangent's own slot of that level where
  // zeros are to be left there afterwards, as the sliding form does, so that the
  // plain adjoint uses no library scratch (callers may have several streams, or be
  // capturing); through scratch where the slots are not to be written.
  const bool slots = gc && zero_s;
  T* scratch = nullptr;
  if (groups.size() > 1 && !slots) {
    int rc = scratch_get(2 * size_t(n) * size_t(count) * sizeof(T), &p);
    if (rc) return rc;
    scratch = static_cast<T*>(p);
  }
  const int64_t per = 2 * n * J;
  const void* in = gy;
  int64_t bs_in = n;
  for (size_t gi = 0; gi < groups.size(); ++gi) {
    const Group& G = groups[gi];
    ModwtArgs a = args_of(G, n);
    a.in = in;
    a.bs_in = bs_in;
    a.xmod = const_cast<void*>(c ? c : gc);
    a.bs_xmod = per;
    q.last = gi + 1 == groups.size();
    if (!q.last) {
      a.out = slots ? static_cast<T*>(gc) + 2 * n * int64_t(G.j0 + G.g - 1)
                    : scratch + int64_t(gi & 1) * n * count;
      a.bs_out = slots ? per : n;
    }
    int rc = modwt_tile_launch<T>(TileOp::kGrad, filt, launch_of(G, count), a, q, st);
    if (rc) return rc;
    in = a.out;
    bs_in = a.bs_out;
  }
  if (slots) {
    int rc = zero_handoffs<T>(gc, groups, n, count, per, st);
    if (rc) return rc;
  }
  if (glam) {
    hipLaunchKernelGGL(grad_sum_k, dim3(unsigned(J)), dim3(256), 0, st, q.partial, glam, count,
                       q.per_signal, gs, q.minlevel, q.maxlevel);
    WH_HIP_CHECK(hipGetLastError());
  }
  return WH_OK;
}

}  // namespace

int modwt_forward(const void* x, void* xmod, int64_t n, int64_t count, int J, int filt,
                  int dtype, hipStream_t st) {
  return dtype == WH_F32 ? modwt_fwd_t<float>(x, xmod, n, count, J, filt, kStoreAll, st)
                         : modwt_fwd_t<double>(x, xmod, n, count, J, filt, kStoreAll, st);
}

int modwt_forward_details(const void* x, void* xmod, int64_t n, int64_t count, int J, int filt,
                          int dtype, hipStream_t st) {
  return dtype == WH_F32 ? modwt_fwd_t<float>(x, xmod, n, count, J, filt, kStoreSmooth, st)
                         : modwt_fwd_t<double>(x, xmod, n, count, J, filt, kStoreSmooth, st);
}

int modwt_inverse(const void* xmod, void* x, int64_t n, int64_t count, int J, int filt, int dtype,
                  const wh_thresh* thr, hipStream_t st, const Candidates& c) {
  return dtype == WH_F32 ? modwt_inv_t<float>(xmod, x, n, count, J, filt, thr, st, nullptr, 0, c)
                         : modwt_inv_t<double>(xmod, x, n, count, J, filt, thr, st, nullptr, 0, c);
}

int modwt_inverse_ws(const void* xmod, void* x, int64_t n, int64_t count, int J, int filt,
                     int dtype, const wh_thresh* thr, void* ws, size_t ws_bytes, hipStream_t st) {
  if (!ws) return set_error(WH_ERR_ARG, "modwt inverse: null workspace");
  return dtype == WH_F32 ? modwt_inv_t<float>(xmod, x, n, count, J, filt, thr, st, ws, ws_bytes)
                         : modwt_inv_t<double>(xmod, x, n, count, J, filt, thr, st, ws, ws_bytes);
}

int modwt_inverse_adjoint(const void* gx, void* gxmod, int64_t n, int64_t count, int J, int filt,
                          int dtype, hipStream_t st) {
  // tiles where the forward runs as tiles (see default_knobs): the same stores bound
  // both.  But one sliding group hands nothing on, so that no slot has to be zeroed
  // afterwards: it keeps what it can fuse beyond a tile group's levels (n = 2^10, J =
  // 9 D4 FP32, three chunks, 8.0 us against 9.9; 256 signals 8.8 against 14.1).
  const size_t esz = dtype == WH_F32 ? 4 : 8;
  const int L = filter_length(filt);
  if (n * count <= (int64_t(1) << 18) && default_knobs(false, n, count, J, filt, esz).first_nt < 0 &&
      (J <= kTileGmax || plan_groups(false, n, J, L, esz, PlanKnobs{}, count).size() > 1))
    return dtype == WH_F32
               ? inv_grad_t<float>(gx, nullptr, gxmod, true, nullptr, n, count, J, filt, nullptr, st)
               : inv_grad_t<double>(gx, nullptr, gxmod, true, nullptr, n, count, J, filt, nullptr,
                                    st);
  return dtype == WH_F32 ? modwt_fwd_t<float>(gx, gxmod, n, count, J, filt, kStoreAdjoint, st)
                         : modwt_fwd_t<double>(gx, gxmod, n, count, J, filt, kStoreAdjoint, st);
}

int modwt_forward_adjoint(const void* gxmod, void* gx, int64_t n, int64_t count, int J, int filt,
                          int dtype, bool details, hipStream_t st) {
  return dtype == WH_F32 ? fwd_adj_t<float>(gxmod, gx, n, count, J, filt, details, st)
                         : fwd_adj_t<double>(gxmod, gx, n, count, J, filt, details, st);
}

int modwt_thresh_inverse_adjoint(const void* gy, const void* c, void* gc, bool zero_s,
                                 double* glam, int64_t n, int64_t count, int J, int filt,
                                 int dtype, const wh_thresh* thr, hipStream_t st) {
  return dtype == WH_F32
             ? inv_grad_t<float>(gy, c, gc, zero_s, glam, n, count, J, filt, thr, st)
             : inv_grad_t<double>(gy, c, gc, zero_s, glam, n, count, J, filt, thr, st);
}

namespace {

template <typename T>
int time_plan(bool inverse, const void* x, void* xmod, void* xr, int64_t n, int J, int filt,
              hipStream_t st, hipEvent_t e0, hipEvent_t e1, float* ms) {
  // an inverse is timed right after a forward, as it runs in a pipeline
  // (the caches then hold what the forward left), a forward after an
  // inverse; the median of the timed runs is kept (a minimum favours plans
  // whose times scatter)
  constexpr int kReps = 9;
  float t_rep[kReps];
  for (int r = 0; r < kReps + 1; ++r) {
    int rc = inverse ? modwt_fwd_t<T>(x, xmod, n, 1, J, filt, kStoreAll, st)
                     : modwt_inv_t<T>(xmod, xr, n, 1, J, filt, nullptr, st);
    if (rc) return rc;
    WH_HIP_CHECK(hipEventRecord(e0, st));
    rc = inverse ? modwt_inv_t<T>(xmod, xr, n, 1, J, filt, nullptr, st)
                 : modwt_fwd_t<T>(x, xmod, n, 1, J, filt, kStoreAll, st);
    if (rc) return rc;
    WH_HIP_CHECK(hipEventRecord(e1, st));
    WH_HIP_CHECK(hipEventSynchronize(e1));
    float t = 0.f;
    WH_HIP_CHECK(hipEventElapsedTime(&t, e0, e1));
    if (r > 0) t_rep[r - 1] = t;  // the first run is a warm-up
  }
  std::sort(t_rep, t_rep + kReps);
  *ms = t_rep[kReps / 2];
  return WH_OK;
}

template <typename T>
int tune_t(int64_t n, int J, int filt, hipStream_t st) {
  const int L = filter_length(filt);
  const size_t esz = sizeof(T);
  void *x = nullptr, *xmod = nullptr, *xr = nullptr;
  auto release = [&] {
    if (x) (void)hipFree(x);
    if (xmod) (void)hipFree(xmod);
    if (xr) (void)hipFree(xr);
  };
  if (hipMalloc(&x, size_t(n) * esz) != hipSuccess ||
      hipMalloc(&xmod, size_t(2) * size_t(n) * size_t(J) * esz) != hipSuccess ||
      hipMalloc(&xr, size_t(n) * esz) != hipSuccess) {
    release();
    return set_error(WH_ERR_NOMEM, "modwt tune: buffer allocation failed");
  }
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = WH_OK;
  hipLaunchKernelGGL(tune_signal_k<T>, dim3(1024), dim3(256), 0, st, static_cast<T*>(x), n);
  hipError_t he = hipGetLastError();
  if (he == hipSuccess) he = hipEventCreate(&e0);
  if (he == hipSuccess) he = hipEventCreate(&e1);
  if (he != hipSuccess) rc = set_hip_error(he, "modwt tune: setup");
  for (int inv = 0; inv < 2 && !rc; ++inv) {
    const bool inverse = inv == 1;
    std::map<std::string, PlanKnobs> cands;  // distinct plans only
    auto add = [&](int g1, int f, int d, int nt) {
      PlanKnobs k;
      k.g1max = g1;
      k.first_per_cu = f;
      k.deep_per_cu = d;
      k.first_nt = nt;
      cands.emplace(plan_text(plan_groups(inverse, n, J, L, esz, k)), k);
    };
    for (int nt : {kNT1, kNT1 / 2}) {
      if (nt == kNT1 / 2 && !inverse) continue;
      for (int g1 = std::min(J, 5); g1 <= kGmax; ++g1)
        for (int f : {1, 2, 4})
          for (int d : {1, 2, 4, 8}) add(g1, f, d, nt);
    }
    for (int nt : {kNT1, kNT1 / 2})  // tiles: only the depth matters
      for (int g1 = 3; g1 <= kTileGmax; ++g1) add(g1, 1, 1, -nt);
    if (inverse && wide_fits(kWideInvP, n, J, esz)) add(kWideGmax, 1, 1, -kWideInvNT);
    // the default plan is timed first and another one is taken only when
    // it is faster by more than the run-to-run spread of these timings
    // (about 1%), so that noise cannot replace the default by a plan that is
    // no better
    constexpr float kMargin = 0.98f;
    const char* env = std::getenv("WH_TUNE_LOG");  // candidate timings to stderr
    const bool log = env && env[0] == '1';
    std::vector<PlanKnobs> order{default_knobs(inverse, n, 1, J, filt, esz)};
    for (auto& c : cands) order.push_back(c.second);
    auto time_knobs = [&](const PlanKnobs& k, float* ms) -> int {
      {
        std::lock_guard<std::mutex> lk(g_knob_mu);
        g_knobs[KnobKey{inv, n, J, filt, int(esz)}] = k;
      }
      const int r = time_plan<T>(inverse, x, xmod, xr, n, J, filt, st, e0, e1, ms);
      if (!r && log)
        std::fprintf(stderr, "wh_modwt_tune %s %.4f ms %s\n", inverse ? "inv" : "fwd", *ms,
                     modwt_plan_string(inverse, n, J, filt, esz == 4 ? WH_F32 : WH_F64).c_str());
      return r;
    };
    float best = 1e30f;
    size_t bi = 0;
    for (size_t i = 0; i < order.size(); ++i) {
      float ms = 0.f;
      if ((rc = time_knobs(order[i], &ms))) break;
      if (i == 0 || ms < best * kMargin) {
        best = ms;
        bi = i;
      }
    }
    // a challenger is confirmed against the default, alternating, so that a
    // drift of the card's speed during the sweep cannot decide the choice
    if (!rc && bi != 0) {
      float tdef[4], tch[4];
      for (int r = 0; r < 4 && !rc; ++r)
        if (!(rc = time_knobs(order[0], &tdef[r]))) rc = time_knobs(order[bi], &tch[r]);
      if (!rc) {
        std::sort(tdef, tdef + 4);
        std::sort(tch, tch + 4);
        if (!(tch[1] + tch[2] < (tdef[1] + tdef[2]) * kMargin)) bi = 0;
      }
    }
    const PlanKnobs bk = order[bi];
    std::lock_guard<std::mutex> lk(g_knob_mu);
    if (rc)
      g_knobs.erase(KnobKey{inv, n, J, filt, int(esz)});
    else
      g_knobs[KnobKey{inv, n, J, filt, int(esz)}] = bk;
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipStreamSynchronize(st);
  release();
  return rc;
}

}  // namespace

int modwt_tune(int64_t n, int J, int filt, int dtype, hipStream_t st) {
  return dtype == WH_F32 ? tune_t<float>(n, J, filt, st) : tune_t<double>(n, J, filt, st);
}

int modwt_force_plan(bool inverse, int64_t n, int J, int filt, int dtype, int g1max,
                     int first_per_cu, int deep_per_cu, int first_nt) {
  const size_t key_esz = dtype == WH_F32 ? 4 : 8;
  const KnobKey key{inverse ? 1 : 0, n, J, filt, int(key_esz)};
  std::lock_guard<std::mutex> lk(g_knob_mu);
  if (g1max <= 0) {
    g_knobs.erase(key);
    return WH_OK;
  }
  if (g1max > kGmax || first_per_cu < 1 || deep_per_cu < 1 ||
      (std::abs(first_nt) != kNT1 && std::abs(first_nt) != kNT1 / 2) ||
      (!inverse && first_nt == kNT1 / 2) || (first_nt < 0 && g1max < 3) ||
      (first_nt < 0 && g1max > kTileGmax &&
       !(inverse && first_nt == -kWideInvNT && wide_fits(kWideInvP, n, J, key_esz))))
    return set_error(WH_ERR_ARG, "modwt plan: knobs out of range");
  PlanKnobs k;
  k.g1max = g1max;
  k.first_per_cu = first_per_cu;
  k.deep_per_cu = deep_per_cu;
  k.first_nt = first_nt;
  g_knobs[key] = k;
  return WH_OK;
}

std::string modwt_plan_string(bool inverse, int64_t n, int J, int filt, int dtype,
                              int64_t count) {
  const int L = filter_length(filt);
  size_t esz = dtype == WH_F32 ? 4 : 8;
  return plan_text(
      plan_groups(inverse, n, J, L, esz, knobs_for(inverse, n, J, filt, esz, count), count));
}

}  // namespace wh
