// batch_plan.hip -- host side of the batched smoothing pipeline: the plan
// (item table, workspace, launch shape), the autotuner and the captured
// graph.  The kernel is in batch_kern.h, instantiated in batch_<type>.hip.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <cmath>
#include <cstdint>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "batch_kern.h"
#include "wh_common.h"
#include "wh_internal.h"

namespace wh {
// Signals smoothed together: as many as the tiles' workspace holds.
struct BatchChunk {
  int item0 = 0, items = 0;  // of the persistent kernel
  int64_t tile0[kBatchPasses] = {};  // per pass
  unsigned tiles[kBatchPasses] = {};
};
}  // namespace wh

struct wh_batch {
  int device = -1;
  int dtype = WH_F64;
  int hardness = 1;
  int count = 0;
  int64_t total = 0;
  std::string key;            // composition signature (tuning table key)
  void* tables = nullptr;          // holds the next four
  wh::BatchItem* items = nullptr;
  wh::BatchTile* tiles = nullptr;  // of the signals that run as tiles
  double* thresh = nullptr;        // one per signal
  int* counter = nullptr;          // queue head, finished workgroups
  void* tscratch = nullptr;        // the tiles' workspace
  size_t tile_bytes = 0;
  std::vector<wh::BatchChunk> chunks;
  void* scratch = nullptr;
  size_t scratch_bytes = 0;
  int64_t stride = 0;         // workspace elements per workgroup
  size_t lds[3] = {0, 0, 0};  // dynamic LDS for 128 / 256 / 512 threads
  int NT = 256;
  unsigned grid = 0;
  int tuned = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
};

namespace wh {
namespace {

constexpr int kNTs[3] = {128, 256, 512};

std::mutex g_tune_mu;
std::map<std::string, std::pair<int, unsigned>> g_tune;  // key -> (NT, grid)

int nt_index(int NT) { return NT == 512 ? 2 : (NT == 256 ? 1 : 0); }

// The tiles' workspace is at most this large (a signal that needs more has a
// chunk of its own): enough that the launches of a chunk fill the chip many
// times over.
constexpr int64_t kBatchTileBytes = int64_t(4) << 30;

// dynamic LDS of one item for NT threads
size_t item_lds(int ttype, int NT, size_t esz) {
  size_t b = (NT == 512) ? block_sel_lds<512>()
             : (NT == 256 ? block_sel_lds<256>() : block_sel_lds<128>());
  b = std::max({b, sel_sampled_lds(NT, esz), sel_small_lds(esz), batch_pre_lds(NT, esz)});
  if (ttype != kDWT) return b;
  const size_t tile = (esz == 8) ? size_t(batch_lds_elems<double>()) * 8
                                 : size_t(batch_lds_elems<float>()) * 4;
  return std::max(b, tile + tile / 2);
}

// shortest DWT signal without tiles that counts as a long walk (see the
// untuned shape in wh_batch_create)
constexpr int kBatchWalk = 1 << 16;

// a DWT signal whose first levels run as tiles
bool dwt_tiled(const BatchItem& I) { return I.n > kBatchDwtWhole && I.J > kBatchHead; }

// The tiles of one signal in a pass; t.kind holds filter and depth.
void add_tiles(std::vector<BatchTile>& tiles, BatchTile t, BatchPass pass) {
  const int J = tile_levels(t.kind), kind = t.kind;
  const bool dwt = kind & kTileDwt;
  const bool last = pass == BatchPass::kDwtLast;
  if (pass != BatchPass::kHead && dwt != last) return;
  if (last || pass == BatchPass::kHead) {
    for (t.m0 = 0; t.m0 < t.n; t.m0 += kBatchP) tiles.push_back(t);
    return;
  }
  const bool second = pass == BatchPass::kSecond;
  if (second && J <= kBatchHead) return;
  const int N = second ? t.n / kBatchRes : t.n, nseq = second ? kBatchRes : 1;
  const int G = second ? J - kBatchHead : std::min(J, kBatchHead);
  const int slots = shrink_slots(second);
  if (N <= slots) {
    const int per = slots / std::max(N, 1 << (G + 1));  // sequences of a tile
    for (int q = 0; q < nseq; q += per) {
      t.kind = kind | q << 8;
      tiles.push_back(t);
    }
    return;
  }
  const int step = slots - 2 * tile_halo(filter_length(kind_filter(kind)), G);
  for (int q = 0; q < nseq; ++q) {
    t.kind = kind | q << 8;
    for (int64_t m = 0; m < N; m += step) {
      t.m0 = int32_t(m);
      tiles.push_back(t);
    }
  }
}

// Chunks, tiles and workspace of a batch's items, longest first.  Signals with
// tiles get their workspace offset and fill the chunks in order; the others
// belong to the first.  Tiles of one filter and depth are neighbours, so that a CU's
// workgroups run the same code.
void plan_chunks(std::vector<BatchItem>& items, std::vector<BatchTile>& tiles,
                 std::vector<BatchChunk>& chunks, int64_t budget, int64_t* workspace) {
  std::vector<std::vector<BatchItem>> by_chunk(1);
  std::vector<std::vector<BatchTile>> heads(1);
  int64_t used = 0;
  size_t expect = 0;  // tiles, about
  *workspace = 0;
  for (BatchItem I : items) {
    I.scr = -1;
    const bool dwt = kind_ttype(I.kind) == kDWT;
    if (dwt && !dwt_tiled(I)) {
      by_chunk[0].push_back(I);
      continue;
    }
    const int64_t need = 3 * batch_pad(I.n);
    if (used && used + need > budget) {
      by_chunk.emplace_back();
      heads.emplace_back();
      used = 0;
    }
    heads.back().push_back(BatchTile{
        I.off, used, I.n, 0, kind_filter(I.kind) | (I.J << 3) | (dwt ? kTileDwt : 0), I.sig});
    I.scr = used;
    by_chunk.back().push_back(I);
    expect += size_t(3 + I.n / (kBatchP / 4));
    used += need;
    *workspace = std::max(*workspace, used);
  }
  items.clear();
  tiles.reserve(expect);
  for (size_t k = 0; k < by_chunk.size(); ++k) {
    BatchChunk c;
    c.item0 = int(items.size());
    c.items = int(by_chunk[k].size());
    items.insert(items.end(), by_chunk[k].begin(), by_chunk[k].end());
    std::stable_sort(heads[k].begin(), heads[k].end(),
                     [](const BatchTile& a, const BatchTile& b) { return a.kind > b.kind; });
    for (int pass = 0; pass < kBatchPasses; ++pass) {
      c.tile0[pass] = int64_t(tiles.size());
      for (const BatchTile& t : heads[k]) add_tiles(tiles, t, BatchPass(pass));
      c.tiles[pass] = unsigned(int64_t(tiles.size()) - c.tile0[pass]);
    }
    chunks.push_back(c);
  }
}

int occupancy(int dtype, int NT, size_t lds, int* blocks) {
  return dtype == WH_F32 ? batch_occupancy<float>(NT, lds, blocks)
                         : batch_occupancy<double>(NT, lds, blocks);
}

// largest resident grid for NT threads
int max_grid(const wh_batch* p, int NT, unsigned* grid, int64_t* resident = nullptr) {
  int occ = 0;
  int rc = occupancy(p->dtype, NT, p->lds[nt_index(NT)], &occ);
  if (rc) return rc;
  if (occ <= 0) return set_error(WH_ERR_UNSUPPORTED, "batch: kernel does not fit a CU");
  const int64_t g = int64_t(occ) * std::max(1, device_info().num_cus);
  *grid = unsigned(std::min<int64_t>(g, p->count));
  if (resident) *resident = g;
  return WH_OK;
}

int ensure_scratch(wh_batch* p, unsigned grid) {
  const size_t esz = p->dtype == WH_F32 ? 4 : 8;
  const size_t need = size_t(grid) * size_t(p->stride) * esz;  // 0: no DWT
  if (need <= p->scratch_bytes) return WH_OK;
  if (p->scratch) {
    WH_HIP_CHECK(hipDeviceSynchronize());
    WH_HIP_CHECK(hipFree(p->scratch));
    p->scratch = nullptr;
    p->scratch_bytes = 0;
  }
  if (hipMalloc(&p->scratch, need) != hipSuccess) {
    p->scratch = nullptr;
    return set_error(WH_ERR_NOMEM, "batch: workspace allocation failed");
  }
  p->scratch_bytes = need;
  return WH_OK;
}

int tile_pass(const wh_batch* p, const BatchChunk& c, BatchPass pass, BatchTileArgs a,
              hipStream_t st) {
  a.tiles = p->tiles + c.tile0[int(pass)];
  const unsigned count = c.tiles[int(pass)];
  return p->dtype == WH_F32 ? batch_tile_launch<float>(pass, count, a, st)
                            : batch_tile_launch<double>(pass, count, a, st);
}

int run(wh_batch* p, int NT, unsigned grid, const void* x, void* y, double* thresh_out,
        hipStream_t st) {
  const size_t esz = p->dtype == WH_F32 ? 4 : 8;
  const char *x0 = static_cast<const char*>(x), *y0 = static_cast<const char*>(y);
  const int64_t bytes = p->total * int64_t(esz);
  BatchTileArgs t{};
  t.x = x;
  t.y = y;
  t.scratch = p->tscratch;
  t.thresh = p->thresh;
  // a tile reads beyond what it writes: overlapping buffers go through a copy
  t.in_place = x0 < y0 + bytes && y0 < x0 + bytes;
  t.hardness = p->hardness;
  for (const BatchChunk& c : p->chunks) {
    if (int rc = tile_pass(p, c, BatchPass::kHead, t, st)) return rc;
    BatchArgs a{};
    a.items = p->items + c.item0;
    a.count = c.items;
    a.counter = p->counter;
    a.x = x;
    a.y = y;
    a.thresh_out = thresh_out;
    a.thresh = p->thresh;
    a.tiles = p->tscratch;
    a.scratch = p->scratch;
    a.scratch_stride = p->stride;
    a.hardness = p->hardness;
    BatchLaunch bl{NT, std::min(grid, unsigned(c.items)), p->lds[nt_index(NT)]};
    if (int rc = p->dtype == WH_F32 ? batch_launch<float>(bl, a, st)
                                    : batch_launch<double>(bl, a, st))
      return rc;
    if (int rc = tile_pass(p, c, BatchPass::kSecond, t, st)) return rc;
    if (int rc = tile_pass(p, c, BatchPass::kFirst, t, st)) return rc;
    if (int rc = tile_pass(p, c, BatchPass::kDwtLast, t, st)) return rc;
  }
  return WH_OK;
}

void drop_graph(wh_batch* p) {
  if (p->gexec) (void)hipGraphExecDestroy(p->gexec);
  if (p->graph) (void)hipGraphDestroy(p->graph);
  p->gexec = nullptr;
  p->graph = nullptr;
}

}  // namespace
}  // namespace wh

using namespace wh;

extern "C" {

int wh_batch_create(const int* lens, const int* filters, const int* ttypes, const int* levels,
                    int count, int dtype, int hardness, wh_batch** out) {
  if (!out) return set_error(WH_ERR_ARG, "null plan pointer");
  *out = nullptr;
  if (!lens || !filters || !ttypes || !levels || count <= 0)
    return set_error(WH_ERR_ARG, "batch: empty or null signal table");
  if (dtype != WH_F64 && dtype != WH_F32) return set_error(WH_ERR_ARG, "bad dtype");
  if (hardness != kHARD && hardness != kSOFT) return set_error(WH_ERR_ARG, "hardness must be 0 or 1");
  int dev = 0;
  WH_HIP_CHECK(hipGetDevice(&dev));
  const size_t esz = dtype == WH_F32 ? 4 : 8;

  std::vector<BatchItem> items(static_cast<size_t>(count));
  std::map<int64_t, int> comp;  // (kind, log2 n, J) -> count
  int64_t off = 0, stride = 0;
  size_t lds[3] = {0, 0, 0};
  for (int i = 0; i < count; ++i) {
    const int64_t n = lens[i];
    const int filt = filters[i], tt = ttypes[i];
    const int L = filter_length(filt);
    if (L == 0) return set_error(WH_ERR_ARG, "batch: filter must be 1..4");
    if (tt != kDWT && tt != kMODWT) return set_error(WH_ERR_ARG, "batch: ttype must be 0 or 1");
    if (n < 2 || (n & (n - 1)) || n > (int64_t(1) << 30))
      return set_error(WH_ERR_ARG, "batch: lengths must be powers of two");
    const int J = resolve_levels(n, levels[i], L);
    if (J <= 0) return set_error(WH_ERR_ARG, "batch: invalid length/levels for the filter");
    if (tt == kMODWT && J > kBatchMaxModwtJ)
      return set_error(WH_ERR_UNSUPPORTED, "batch: MODWT depth above 8 (use wh_smooth)");
    BatchItem& I = items[size_t(i)];
    I.off = off;
    I.n = int32_t(n);
    I.J = J;
    I.kind = batch_kind(tt, filt);
    I.sig = i;
    // factor of univ_thresh(w, 0, 0) (src/thresh.cpp:170-201): a one-level
    // DWT takes the MAD of x[1..n-1] scaled by sqrt(2 ln(n-1))
    const double nn = (tt == kDWT && J == 1) ? double(n - 1) : double(n);
    I.factor = std::sqrt(2.0 * std::log(nn));
    off += n;
    if (tt == kDWT) stride = std::max<int64_t>(stride, 2 * (dwt_tiled(I) ? n >> kBatchHead : n));
    for (int k = 0; k < 3; ++k) lds[k] = std::max(lds[k], item_lds(tt, kNTs[k], esz));
    int lg = 0;
    while ((int64_t(1) << lg) < n) ++lg;
    comp[(int64_t(I.kind) << 16) | (lg << 8) | J] += 1;
  }
  // longest work first within a chunk: the selection passes over D_1, the
  // DWT's levels move about 6 words per sample plus their serial latency
  auto cost = [](const BatchItem& I) {
    if (kind_ttype(I.kind) == kMODWT) return int64_t(I.n) * 2;
    if (dwt_tiled(I)) return int64_t(I.n) + (int64_t(I.n) >> kBatchHead) * 6 + 256 * I.J;
    return int64_t(I.n) * 6 + 256 * I.J;
  };
  std::stable_sort(items.begin(), items.end(),
                   [&](const BatchItem& a, const BatchItem& b) { return cost(a) > cost(b); });
  const double max_cost = double(cost(items[0]));
  double sum_cost = 0.0, walk_cost = 0.0;  // walk: long DWT signals without tiles
  for (const BatchItem& I : items) {
    sum_cost += double(cost(I));
    if (kind_ttype(I.kind) == kDWT && !dwt_tiled(I) && I.n >= kBatchWalk) walk_cost += double(cost(I));
  }
  std::vector<BatchTile> tiles;
  std::vector<BatchChunk> chunks;
  int64_t tscr = 0;  // elements of the tiles' workspace
  plan_chunks(items, tiles, chunks, int64_t(kBatchTileBytes / int64_t(esz)), &tscr);

  wh_batch* p = new wh_batch();
  p->device = dev;
  p->dtype = dtype;
  p->hardness = hardness;
  p->count = count;
  p->chunks = std::move(chunks);
  p->total = off;
  p->stride = (stride + 63) / 64 * 64;
  for (int k = 0; k < 3; ++k) p->lds[k] = lds[k];
  p->key = std::to_string(dtype) + "/" + std::to_string(hardness) + ":";
  for (auto& kv : comp) p->key += std::to_string(kv.first) + "x" + std::to_string(kv.second) + ",";

  auto fail = [&](int rc) {
    wh_batch_destroy(p);
    return rc;
  };
  // the device tables in one allocation: items, the queue's two zeros, room for the
  // thresholds, tiles.  What is small goes up in one copy (an allocation or a copy
  // costs a plan of a few short signals as much as the rest of its creation); the
  // tiles of a large batch are not copied once more for it.
  const size_t item_bytes = sizeof(BatchItem) * size_t(count), head_bytes = item_bytes + 8;
  const size_t list_at = head_bytes + sizeof(double) * size_t(count);
  const size_t list_bytes = sizeof(BatchTile) * tiles.size();
  static_assert(sizeof(BatchItem) % 8 == 0 && 2 * sizeof(int) == 8, "tables stay aligned");
  const bool one = list_at + list_bytes <= (size_t(1) << 16);
  std::vector<unsigned char> up(one ? list_at + list_bytes : head_bytes);
  std::memcpy(up.data(), items.data(), item_bytes);
  if (one && list_bytes) std::memcpy(up.data() + list_at, tiles.data(), list_bytes);
  if (hipMalloc(&p->tables, list_at + list_bytes) != hipSuccess) {
    p->tables = nullptr;
    return fail(set_error(WH_ERR_NOMEM, "batch: table allocation failed"));
  }
  unsigned char* at = static_cast<unsigned char*>(p->tables);
  p->items = reinterpret_cast<BatchItem*>(at);
  p->counter = reinterpret_cast<int*>(at + item_bytes);
  p->thresh = reinterpret_cast<double*>(at + head_bytes);
  p->tiles = reinterpret_cast<BatchTile*>(at + list_at);
  if (hipMemcpy(at, up.data(), up.size(), hipMemcpyHostToDevice) != hipSuccess ||
      (!one && list_bytes &&
       hipMemcpy(at + list_at, tiles.data(), list_bytes, hipMemcpyHostToDevice) != hipSuccess))
    return fail(set_hip_error(hipGetLastError(), "batch: table upload"));
  p->tile_bytes = size_t(tscr) * esz;
  if (p->tile_bytes && hipMalloc(&p->tscratch, p->tile_bytes) != hipSuccess) {
    p->tscratch = nullptr;
    return fail(set_error(WH_ERR_NOMEM, "batch: workspace allocation failed"));
  }

  // the persistent kernel's shape: a tuned one for this composition, or
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune.find(p->key);
    if (it != g_tune.end()) {
      p->NT = it->second.first;
      p->grid = it->second.second;
      p->tuned = 1;
    }
  }
  if (!p->tuned) {
    // untuned: 256 threads and every workgroup that fits, unless the longest
    // item would still run when the others are done: then 512 threads, which
    // take it in about two thirds of the time.  Mixed batches, us with 256 /
    // 512 threads: 8192 signals to 2^16 samples FP64 2188 / 2453, FP32 1382 /
    // 1637; 2000 to 2^16 FP64 629 / 620; 1200 to 2^16 (0.27 where the line is
    // 0.4) FP64 445 / 376, FP32 296 / 257; 300 to 2^16 FP64 256 / 156.  512
    // threads also where most of the work is long DWT signals without tiles,
    // whose walk through memory gains nothing from a third workgroup a CU (J = 3,
    // 1024 x 2^17 FP64 1942 / 1789, FP32 1235 / 1081; 1024 x 2^16 976 / 880 and 629 /
    // 494; of 2^14, 4096 825 / 902 and 487 / 654).  wh_batch_tune times the shapes.
    int64_t resident = 0;
    p->NT = 256;
    if (int rc = max_grid(p, p->NT, &p->grid, &resident)) return fail(rc);
    if (sum_cost < 0.4 * max_cost * double(resident) || walk_cost > 0.5 * sum_cost) {
      p->NT = 512;
      if (int rc = max_grid(p, p->NT, &p->grid)) return fail(rc);
    }
  }
  if (int rc = ensure_scratch(p, p->grid)) return fail(rc);
  *out = p;
  return WH_OK;
}

void wh_batch_destroy(wh_batch* p) {
  if (!p) return;
  (void)hipDeviceSynchronize();
  drop_graph(p);
  if (p->tables) (void)hipFree(p->tables);
  if (p->tscratch) (void)hipFree(p->tscratch);
  if (p->scratch) (void)hipFree(p->scratch);
  delete p;
}

// the packed signals start at even offsets; the kernels move element pairs
// with single vector accesses, so the buffers must be aligned to two elements
static int check_io(const wh_batch* p, const void* x, const void* y) {
  if (!p || !x || !y) return set_error(WH_ERR_ARG, "null pointer");
  const uintptr_t pair = p->dtype == WH_F64 ? 16 : 8;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & (pair - 1))
    return set_error(WH_ERR_ARG, "device buffers must be aligned to two elements (16 bytes FP64, 8 bytes FP32)");
  return WH_OK;
}

int wh_batch_smooth(wh_batch* p, const void* x, void* y, double* thresh_out, void* stream) {
  if (int rc = check_io(p, x, y)) return rc;
  return run(p, p->NT, p->grid, x, y, thresh_out, static_cast<hipStream_t>(stream));
}

int wh_batch_tune(wh_batch* p, const void* x, void* y, double* thresh_out, void* stream) {
  if (int rc = check_io(p, x, y)) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int cus = std::max(1, device_info().num_cus);
  struct Cand {
    int NT;
    unsigned grid;
  };
  std::vector<Cand> cands;
  unsigned gmax_all = 0;
  for (int NT : kNTs) {
    unsigned gmax = 0;
    if (int rc = max_grid(p, NT, &gmax)) return rc;
    gmax_all = std::max(gmax_all, gmax);
    for (unsigned g = unsigned(cus); g < gmax; g += unsigned(cus)) cands.push_back({NT, g});
    cands.push_back({NT, gmax});
  }
  if (int rc = ensure_scratch(p, gmax_all)) return rc;
  hipEvent_t e0, e1;
  WH_HIP_CHECK(hipEventCreate(&e0));
  WH_HIP_CHECK(hipEventCreate(&e1));
  float best = 1e30f;
  Cand bc = {p->NT, p->grid};
  int rc = WH_OK;
  const bool log = std::getenv("WH_TUNE_LOG") != nullptr;  // candidate timings to stderr
  for (const Cand& c : cands) {
    if ((rc = run(p, c.NT, c.grid, x, y, thresh_out, st))) break;  // warm-up
    float tmin = 1e30f;
    for (int r = 0; r < 3 && !rc; ++r) {
      if (hipEventRecord(e0, st) != hipSuccess) rc = set_hip_error(hipGetLastError(), "event");
      if (!rc) rc = run(p, c.NT, c.grid, x, y, thresh_out, st);
      if (!rc && hipEventRecord(e1, st) != hipSuccess) rc = set_hip_error(hipGetLastError(), "event");
      if (!rc && hipEventSynchronize(e1) != hipSuccess) rc = set_hip_error(hipGetLastError(), "sync");
      float ms = 0.f;
      if (!rc && hipEventElapsedTime(&ms, e0, e1) == hipSuccess) tmin = std::min(tmin, ms);
    }
    if (rc) break;
    if (log) std::fprintf(stderr, "wh_batch_tune: %d threads x %u workgroups: %.3f ms\n", c.NT, c.grid, tmin);
    if (tmin < best) {
      best = tmin;
      bc = c;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) return rc;
  p->NT = bc.NT;
  p->grid = bc.grid;
  p->tuned = 1;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tune[p->key] = {p->NT, p->grid};
  }
  drop_graph(p);
  // leave y holding the result of the chosen shape
  return run(p, p->NT, p->grid, x, y, thresh_out, st);
}

int wh_batch_capture(wh_batch* p, const void* x, void* y, double* thresh_out) {
  if (int rc = check_io(p, x, y)) return rc;
  drop_graph(p);
  hipStream_t cs;
  WH_HIP_CHECK(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
  int rc = WH_OK;
  if (hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) != hipSuccess) {
    rc = set_hip_error(hipGetLastError(), "hipStreamBeginCapture");
  } else {
    rc = run(p, p->NT, p->grid, x, y, thresh_out, cs);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(cs, &g);
    if (!rc && e != hipSuccess) rc = set_hip_error(e, "hipStreamEndCapture");
    if (!rc) {
      hipGraphExec_t ge = nullptr;
      e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
      if (e != hipSuccess) {
        rc = set_hip_error(e, "hipGraphInstantiate");
        (void)hipGraphDestroy(g);
      } else {
        p->graph = g;
        p->gexec = ge;
      }
    } else if (g) {
      (void)hipGraphDestroy(g);
    }
  }
  (void)hipStreamDestroy(cs);
  return rc;
}

int wh_batch_replay(wh_batch* p, void* stream) {
  if (!p) return set_error(WH_ERR_ARG, "null pointer");
  if (!p->gexec) return set_error(WH_ERR_ARG, "batch: no captured graph");
  WH_HIP_CHECK(hipGraphLaunch(p->gexec, static_cast<hipStream_t>(stream)));
  return WH_OK;
}

int wh_batch_info(const wh_batch* p, int64_t* total, int* threads, int* workgroups,
                  int64_t* lds_bytes, int64_t* workspace_bytes, int* tuned) {
  if (!p) return set_error(WH_ERR_ARG, "null pointer");
  if (total) *total = p->total;
  if (threads) *threads = p->NT;
  if (workgroups) *workgroups = int(p->grid);
  if (lds_bytes) *lds_bytes = int64_t(p->lds[nt_index(p->NT)]);
  if (workspace_bytes) *workspace_bytes = int64_t(p->scratch_bytes + p->tile_bytes);
  if (tuned) *tuned = p->tuned;
  return WH_OK;
}

int wh_debug_batch_set_shape(wh_batch* p, int threads, int workgroups) {
  if (!p) return set_error(WH_ERR_ARG, "null plan");
  if (threads != 128 && threads != 256 && threads != 512)
    return set_error(WH_ERR_ARG, "batch: threads must be 128, 256 or 512");
  unsigned gmax = 0;
  if (int rc = max_grid(p, threads, &gmax)) return rc;
  if (workgroups < 1 || unsigned(workgroups) > gmax)
    return set_error(WH_ERR_ARG, "batch: workgroups must be 1..the resident maximum");
  if (int rc = ensure_scratch(p, unsigned(workgroups))) return rc;
  p->NT = threads;
  p->grid = unsigned(workgroups);
  drop_graph(p);
  return WH_OK;
}

}  // extern "C"
