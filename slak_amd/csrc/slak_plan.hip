// Level plans over a union of meshes (see slak_plan.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "slak_plan.hpp"

namespace slak {

std::string flags_message(int f) {
  std::string m;
  if (f & kFlagBadPtr) m += " ptr is not a valid CSR offset array (ptr[0]=0, non-decreasing, ptr[nf]=nnz);";
  if (f & kFlagBadOrder) m += " face with fewer than three vertices;";
  if (f & kFlagBadId) m += " vertex id out of range;";
  if (f & kFlagBadVals) m += " vals is not a permutation of 1..face order;";
  if (f & kFlagBadQuad) m += " QUAD mesh with a face that is not a quad at ptr = 4i;";
  if (f & kFlagDupHalfEdge)
    m += " non-manifold: a directed edge occurs twice (inconsistent orientation or >2 faces on an edge);";
  if (f & kFlagDegenerate) m += " degenerate face (repeated vertex along a face);";
  if (f & kFlagOverflow) m += " index overflow (counts exceed int32);";
  if (f & kFlagChanged) m += " the number of edges differs from the one the batch was created with;";
  return m;
}

namespace {

constexpr int kReportAt = 32;  // ints: the late flags word has a line of its own

int64_t* pinned_buffer(size_t n) {
  struct Pinned {
    int64_t* p = nullptr;
    size_t n = 0;
    ~Pinned() {
      if (p) (void)hipHostFree(p);
    }
  };
  thread_local Pinned pin;
  if (pin.n < n) {
    if (pin.p) (void)hipHostFree(pin.p);
    pin.p = nullptr;
    pin.n = 0;
    SLAK_HIP_CHECK(hipHostMalloc((void**)&pin.p, n * sizeof(int64_t)));
    pin.n = n;
  }
  return pin.p;
}

// Pinned host blocks for table uploads, by power-of-two size class (4 KiB
// and up): a pageable source makes hipMemcpyAsync stage the bytes itself
// before it returns, which delays every launch queued after it.
std::mutex g_pin_mu;
std::vector<std::pair<size_t, char*>> g_pin_free;

char* pinned_acquire(size_t bytes, size_t& cap) {
  cap = 4096;
  while (cap < bytes) cap <<= 1;
  {
    std::lock_guard<std::mutex> g(g_pin_mu);
    for (size_t i = 0; i < g_pin_free.size(); ++i)
      if (g_pin_free[i].first == cap) {
        char* p = g_pin_free[i].second;
        g_pin_free[i] = g_pin_free.back();
        g_pin_free.pop_back();
        return p;
      }
  }
  char* p = nullptr;
  SLAK_HIP_CHECK(hipHostMalloc((void**)&p, cap));
  return p;
}

void pinned_release(char* p, size_t cap) {
  if (!p) return;
  std::lock_guard<std::mutex> g(g_pin_mu);
  if (g_pin_free.size() < 64) {
    g_pin_free.emplace_back(cap, p);
    return;
  }
  (void)hipHostFree(p);
}

void check_i32(int64_t x, const std::string& what) {
  if (x < 0 || x > 0x7fffffffll)
    throw Error(SLAK_ERR_INVALID_ARGUMENT, "too large for int32 indices: " + what + " = " + std::to_string(x));
}

}  // namespace

// Register capacity of the first level's row kernels: rows up to it are
// processed in registers, longer ones (correct for any length, slower) from
// memory. SLAK_ROW_CAP=4 sends rows of 5 and more down the in-memory path.
static int row_capacity() {
  const char* e = std::getenv("SLAK_ROW_CAP");
  return e && std::atoi(e) == 4 ? 4 : kRowSlots;
}

// Rows per block and LDS row tile of the first level's numbering. A block of
// R rows needs about R m + 3 sqrt(R) sigma tile entries, with m the mean row
// length (corners over vertices) and sigma the spread of row lengths from the
// histogram (hist: kRowHistBins counts, the last bin "longer"; without one,
// sigma = 1): R is the largest of 256, 128, 64 whose need fits kRowTileMax
// (half of it when rows average more than 5), and the tile that need rounded
// up to 256 entries (at least 1024). A block whose rows exceed the tile stores
// them directly. SLAK_ROWS_PER_BLOCK forces R.
RowTiling autotune_rows(int64_t nv, int64_t nnz, const int64_t* hist) {
  double m = nv > 0 ? (double)nnz / (double)nv : 4.0;
  double sigma = 1.0;
  if (hist) {
    double n = 0, sq = 0;
    for (int b = 0; b < kRowHistBins; ++b) {
      n += (double)hist[b];
      sq += (double)hist[b] * (b - m) * (b - m);
    }
    if (n > 0) sigma = std::sqrt(sq / n);
  }
  auto need = [&](int R) { return R * m + 3.0 * std::sqrt((double)R) * sigma; };
  int R = 64;
  for (int r : {256, 128})
    if (need(r) <= (double)kRowTileMax) {
      R = r;
      break;
    }
  if (m > 5.0) R = std::max(64, R / 2);
  if (const char* e = std::getenv("SLAK_ROWS_PER_BLOCK")) {
    const int forced = std::atoi(e);
    if (forced == 64 || forced == 128 || forced == 256) R = forced;
  }
  const double want = std::ceil(need(R) / 256.0) * 256.0;
  return RowTiling{R, (int)std::min<double>(kRowTileMax, std::max(1024.0, want))};
}

Plan::Plan(int scheme, std::vector<MeshJob> jobs, OutputMode mode, hipStream_t st)
    : scheme_(scheme), jobs_(std::move(jobs)), mode_(mode), st_(st), arena_(pool()) {
  init_device_options();
}

Plan::~Plan() {
  if (exec_) (void)hipGraphExecDestroy(exec_);
  if (graph_) (void)hipGraphDestroy(graph_);
  if (owned_st_) {
    (void)hipStreamSynchronize(owned_st_);
    (void)hipStreamDestroy(owned_st_);
    (void)hipEventDestroy(order_ev_);
  }
  bool held = false;
  for (auto& j : jobs_) held |= j.out_ids != nullptr;
  if (!outputs_released_ && held) {
    (void)hipStreamSynchronize(st_);
    if (mode_ == OutputMode::kSeparate)
      for (auto& j : jobs_)
        for (void* p : {(void*)j.out_verts, (void*)j.out_ids, (void*)j.out_ptr, (void*)j.out_vals})
          if (p) pool().release(p);
  }
  if (!arena_.empty() || staging_first_.p || staging_all_.p || host_words_.p) (void)hipStreamSynchronize(st_);
  pinned_release(staging_first_.p, staging_first_.cap);
  pinned_release(staging_all_.p, staging_all_.cap);
  pinned_release(host_words_.p, host_words_.cap);
}

// The device's flags word, after everything queued on the plan's stream.
int Plan::read_flags() {
  int32_t* pin = reinterpret_cast<int32_t*>(pinned_buffer(1));
  SLAK_HIP_CHECK(hipMemcpyAsync(pin, d_flags_, sizeof(int32_t), hipMemcpyDeviceToHost, st_));
  SLAK_HIP_CHECK(hipStreamSynchronize(st_));
  ++syncs_;
  return *pin;
}

// Waits until the analysis has filled the report. The host looks at the done
// word itself (an event wait returns about 5 us later); now and then it asks
// for the stream's state, which ends the wait if the work has failed.
void Plan::wait_report() {
  auto done = [this] { return __atomic_load_n(report_, __ATOMIC_ACQUIRE) != 0; };
  for (int64_t i = 1; !done(); ++i) {
    if (i % 4096) continue;
    const hipError_t e = hipStreamQuery(st_);
    if (e == hipErrorNotReady) continue;
    if (e != hipSuccess) SLAK_HIP_CHECK(e);
    if (!done()) throw Error(SLAK_ERR_INTERNAL, "the analysis ended without its report");
  }
  ++syncs_;
}

// Uploads the segment tables (SegDesc, vertex, face and corner bases, first
// segment of every block) of levels [l0, l1) in one copy from a plan-owned staging buffer (one per call site,
// so a pending copy never sees its source rewritten).
void Plan::upload_tables(int l0, int l1, Staging& staging, bool zero_state) {
  auto align = [](size_t x) { return (x + 255) & ~(size_t)255; };
  size_t total = 0;
  std::vector<size_t> offs;
  // k_final tables of several meshes: FinalSeg[n] and the mesh of every block
  auto table_bytes = [&](const FinalTable& T) -> size_t {
    return final_table(T) ? align(T.segs.size() * sizeof(FinalSeg)) + align(T.block_seg.size() * sizeof(int32_t)) : 0;
  };
  auto fin_bytes = [&](const LevelPlan& L) -> size_t {
    return table_bytes(L.fin) + table_bytes(L.pos) + table_bytes(L.deep);
  };
  // a level of one mesh is described in its launches' arguments
  auto nblocks = [](int64_t items) { return (size_t)((items + kBlockItems - 1) / kBlockItems); };
  for (int l = l0; l < l1; ++l) {
    const LevelPlan& L = levels_[l];
    const size_t n = L.segs.size();
    offs.push_back(total);
    if (n > 1) total = align(total + n * sizeof(SegDesc));
    if (n > 1 && !L.d_vblk)  // (the first level's second upload changes its descriptors alone)
      total += align(3 * (n + 1) * sizeof(int64_t)) +
               align((nblocks(L.nv) + nblocks(L.nf) + nblocks(L.nnz) + 3) * sizeof(int32_t));
    total += fin_bytes(L);
  }
  // (planned with the last levels: empty when the first level's tables go up)
  const size_t lak_bytes = lak_.segs.empty() ? 0 : align(lak_.segs.size() * sizeof(LakSeg)) + align(lak_.block_seg.size() * sizeof(int32_t));
  total += lak_bytes;
  for (int l = l0; l < l1; ++l)
    if (!levels_[l].d_mflags)
      levels_[l].d_mflags = l == 0 ? d_state_ + kStateBounds + (levels_[l].segs.size() + 1)
                                   : arena_.get_n<int>((int64_t)std::max<size_t>(levels_[l].segs.size(), 1));
  if (total == 0) {
    if (zero_state) launch_setup(nullptr, nullptr, 0, d_state_, n_state_, st_);
    return;
  }
  if (staging.p) SLAK_HIP_CHECK(hipStreamSynchronize(st_));  // reused: an earlier copy may still read it
  if (staging.cap < total) {
    pinned_release(staging.p, staging.cap);
    staging.p = pinned_acquire(total, staging.cap);
  }
  char* d = arena_.get_n<char>((int64_t)total);
  for (int l = l0; l < l1; ++l) {
    LevelPlan& L = levels_[l];
    const size_t n = L.segs.size();
    size_t o = offs[l - l0];
    if (n > 1) {
      std::memcpy(staging.p + o, L.segs.data(), n * sizeof(SegDesc));
      L.d_segs = reinterpret_cast<SegDesc*>(d + o);
      o = align(o + n * sizeof(SegDesc));
    }
    if (n > 1 && !L.d_vblk) {
      const std::vector<int64_t>* bases[3] = {&L.vbase, &L.fbase, &L.cbase};
      int64_t** d_bases[3] = {&L.d_vbase, &L.d_fbase, &L.d_cbase};
      for (int i = 0; i < 3; ++i) {
        std::memcpy(staging.p + o + i * (n + 1) * sizeof(int64_t), bases[i]->data(), (n + 1) * sizeof(int64_t));
        *d_bases[i] = reinterpret_cast<int64_t*>(d + o) + i * (n + 1);
      }
      o = align(o + 3 * (n + 1) * sizeof(int64_t));
      // the mesh of each block's first item
      int32_t** d_blks[3] = {&L.d_vblk, &L.d_fblk, &L.d_cblk};
      size_t at = 0;
      for (int i = 0; i < 3; ++i) {
        int32_t* blk = reinterpret_cast<int32_t*>(staging.p + o) + at;
        *d_blks[i] = reinterpret_cast<int32_t*>(d + o) + at;
        const std::vector<int64_t>& base = *bases[i];
        const size_t nb = nblocks(base.back());
        for (size_t k = 0; k < n; ++k) std::fill(blk + nblocks(base[k]), blk + nblocks(base[k + 1]), (int32_t)k);
        blk[nb] = (int32_t)n - 1;
        at += nb + 1;
      }
      o = align(o + at * sizeof(int32_t));
    }
    for (FinalTable* T : {&L.fin, &L.pos, &L.deep}) {
      if (!final_table(*T)) continue;
      std::memcpy(staging.p + o, T->segs.data(), T->segs.size() * sizeof(FinalSeg));
      T->d_segs = reinterpret_cast<FinalSeg*>(d + o);
      o = align(o + T->segs.size() * sizeof(FinalSeg));
      const size_t nb = T->block_seg.size() * sizeof(int32_t);
      std::memcpy(staging.p + o, T->block_seg.data(), nb);
      T->d_block_seg = reinterpret_cast<int32_t*>(d + o);
      o = align(o + nb);
    }
  }
  if (lak_bytes) {
    size_t o = total - lak_bytes;
    std::memcpy(staging.p + o, lak_.segs.data(), lak_.segs.size() * sizeof(LakSeg));
    lak_.d_segs = reinterpret_cast<LakSeg*>(d + o);
    o = align(o + lak_.segs.size() * sizeof(LakSeg));
    std::memcpy(staging.p + o, lak_.block_seg.data(), lak_.block_seg.size() * sizeof(int32_t));
    lak_.d_block_seg = reinterpret_cast<int32_t*>(d + o);
  }
  launch_setup(staging.p, d, (int64_t)total, zero_state ? d_state_ : nullptr, zero_state ? n_state_ : 0, st_);
}

std::string Plan::describe_failure(int fl) const {
  std::string m;
  for (size_t j = 0; j < jobs_.size(); ++j)
    if (jobs_[j].bad_flags) {
      m = "mesh " + std::to_string(j) + ":" + flags_message(jobs_[j].bad_flags);
      break;
    }
  if (m.empty()) m = flags_message(fl);
  return "invalid mesh: " + m;
}

// First level: per-job bases, the caller meshes gathered into the union.
void Plan::plan_first_level() {
  levels_.clear();
  levels_.emplace_back();
  LevelPlan& L = levels_[0];
  bool all_quad = true;
  for (size_t j = 0; j < jobs_.size(); ++j) {
    MeshJob& J = jobs_[j];
    if (J.levels <= 0) continue;
    all_quad &= J.in.type == SLAK_QUAD;
  }
  L.quad = all_quad;
  int64_t vb = 0, fb = 0, cb = 0;
  for (size_t j = 0; j < jobs_.size(); ++j) {
    MeshJob& J = jobs_[j];
    if (J.levels <= 0) continue;
    SegDesc S{};
    S.vb = vb;
    S.fb = fb;
    S.cb = cb;
    S.nv = (int32_t)J.in.nverts;
    S.nf = (int32_t)J.in.nfaces;
    S.nnz = (int64_t)J.in.nnz;
    S.src_ptr = J.in.ptr;
    S.src_ids = J.in.ids;
    S.src_vals = J.in.vals;
    S.src_verts = reinterpret_cast<const float4*>(J.in.verts);
    S.src_stride = J.in.ptr ? 0 : (J.in.type == SLAK_QUAD ? 4 : 3);
    S.require_quad = J.in.type == SLAK_QUAD;
    L.jobs.push_back((int)j);
    L.segs.push_back(S);
    L.vbase.push_back(vb);
    L.fbase.push_back(fb);
    L.cbase.push_back(cb);
    vb += S.nv;
    fb += S.nf;
    cb += S.nnz;
  }
  L.vbase.push_back(vb);
  L.fbase.push_back(fb);
  L.cbase.push_back(cb);
  L.nv = vb;
  L.nf = fb;
  L.nnz = cb;
  check_i32(L.nv, "vertices of the first level");
  check_i32(L.nf, "faces of the first level");
  check_i32(L.nnz, "corners of the first level");
  check_i32(4 * L.nnz, "refined corners of the first level");
  const RowTiling rt = autotune_rows(L.nv, L.nnz, nullptr);
  L.cap = row_capacity();
  L.rows = rt.rows;
  L.tile = rt.tile;

  // one arena block for the first level's buffers and the analysis state
  // that follows (the table upload, the scan partials, a single mesh's
  // boundary flags); anything beyond it comes from the pool as before
  const int64_t nseg = (int64_t)L.segs.size();
  const int64_t at_dev = (kStateBounds + 2 * nseg + 1 + 3) & ~(int64_t)3;  // 16-byte aligned
  const int64_t ntiles = (L.nv + kBlockItems - 1) / kBlockItems, ngroups = (ntiles + kTilesPerGroup - 1) / kTilesPerGroup;
  const int64_t at_groups = at_dev + 4;
  const int64_t at_cnt = (at_groups + 2 * ngroups + 3) & ~(int64_t)3;
  n_state_ = (at_cnt + L.nv + 3) & ~(int64_t)3;
  {
    auto line = [](int64_t n, size_t elem) { return ((size_t)std::max<int64_t>(n, 1) * elem + 255) & ~(size_t)255; };
    size_t est = 2 * line(L.nnz, 4) + 2 * line(L.nnz, 8) + line(L.nv, 4 * kRowSlots) + 2 * line(L.nv, 4) +
                 2 * line(L.nv + 1, 4) + line(n_state_, 4) +
                 line(ntiles, 8);
    if (!L.quad) est += line(L.nf + 1, 4) + line(L.nnz, 4);
    if (L.segs.size() != 1) est += line(L.nv, 16);
    if (scheme_ == kSLAK) est += line(L.nnz, 4);
    est += (size_t)256 << 10;
    arena_.reserve(est);
  }
  int32_t* ids_pos = arena_.get_n<int32_t>(L.nnz);
  L.ids = ids_pos;
  if (!L.quad) {
    L.fptr = arena_.get_n<int32_t>(L.nf + 1);
    L.cface = arena_.get_n<int32_t>(L.nnz);
  }
  if (L.segs.size() == 1) {
    L.P = L.segs[0].src_verts;
  } else {
    P1_ = arena_.get_n<float4>(L.nv);
    L.P = P1_;
  }
  d_state_ = arena_.get_n<int32_t>(n_state_);
  d_flags_ = d_state_;
  L.pool = d_state_ + at_dev;
  L.group_sum = reinterpret_cast<uint64_t*>(d_state_ + at_groups);
  n_groups_ = ngroups;
  L.cnt = d_state_ + at_cnt;
  L.slots = arena_.get_n<int32_t>(kRowSlots * L.nv);
  L.head = arena_.get_n<int32_t>(L.nv);
  L.ecnt = arena_.get_n<int32_t>(L.nv);
  L.tile_sum = arena_.get_n<uint64_t>(ntiles);
  L.tptr = arena_.get_n<int32_t>(L.nv + 1);
  L.tids = arena_.get_n<int32_t>(L.nnz);
  L.trow = arena_.get_n<int2>(L.nnz);
  L.ci = arena_.get_n<int2>(L.nnz);
  if (scheme_ == kSLAK) L.mpos = arena_.get_n<int32_t>(L.nnz);
  L.eptr = arena_.get_n<int32_t>(L.nv + 1);
}

LevelView LevelPlan::view(int* flags, int* late) const {
  LevelView V{};
  V.ids = ids;
  V.fptr = fptr;
  V.cface = cface;
  V.P = P;
  V.nv = (int32_t)nv;
  V.nf = (int32_t)nf;
  V.nnz = nnz;
  V.tptr = tptr;
  V.cnt = cnt;
  V.slots = slots;
  V.head = head;
  V.next = reinterpret_cast<int32_t*>(ci);  // free until the numbering writes the pairs
  V.tids = tids;
  V.pool = pool;
  V.ecnt = ecnt;
  V.tile_sum = tile_sum;
  V.group_sum = group_sum;
  V.row_cap = cap;
  V.rows_per_block = rows;
  V.trow = trow;
  V.mpos = mpos;
  V.eptr = eptr;
  V.flags = flags;
  V.late = late;
  V.seg = table();
  V.tile_entries = tile;
  return V;
}

// Validation, position order, valences and the rows' corners in one launch.
void Plan::record_gather(LevelPlan& L) {
  ProfScope ps(st_, {"gather", gather_bytes(L)}, gather_stages(L));
  launch_gather(L.quad, L.table(), scheme_ == kLAK, const_cast<int32_t*>(L.ids), L.view(d_flags_, late_), st_);
}

// First-level analysis: sorted rows of M^T with in-neighbours and their
// offsets, owned-edge counts and offsets (later levels receive their structure
// from the level before).
void Plan::record_analysis(LevelPlan& L) {
  LevelView V = L.view(d_flags_, late_);
  V.hist_rows = d_state_ + kStateRowHist;
  V.bounds = d_state_ + kStateBounds;
  V.planned = replayed_ ? 1 : 0;
  // reads the rows and their corners' neighbours, writes the owned counts
  ProfScope ps(st_, {L.quad ? "symbolic_quad" : "symbolic_poly",
                     8.0 * L.nnz + 8.0 * L.nv + (L.quad ? 0.0 : 4.0 * L.nnz + 4.0 * (L.nf + 1))},
               analysis_stages(L));
  launch_symbolic(L.quad, scheme_, V, st_);
  if (L.segs.size() > 1) launch_seg_bounds(V, st_);
}

// reads face offsets, ids and vals, writes the ids in position order, the
// rows' corners and the valences (polygons: face offsets and corner faces)
double Plan::gather_bytes(const LevelPlan& L) const {
  return 4.0 * (L.nf + 1) + 16.0 * L.nnz + 4.0 * L.nv + (L.quad ? 0.0 : 4.0 * L.nnz + 4.0 * (L.nf + 1));
}

std::vector<StageBytes> Plan::gather_stages(const LevelPlan& L) const {
  return {{"gather", 4.0 * (L.nf + 1) + 12.0 * L.nnz + (L.quad ? 0.0 : 8.0 * L.nnz + 4.0 * L.nf)},
          {L.quad ? "count_quad" : "count_poly", 4.0 * L.nnz + 8.0 * L.nv + (L.quad ? 0.0 : 4.0 * L.nf)},
          {L.quad ? "transpose_quad" : "transpose_poly", 8.0 * L.nnz + 12.0 * L.nv + (L.quad ? 0.0 : 4.0 * L.nf)}};
}

std::vector<StageBytes> Plan::analysis_stages(const LevelPlan& L) const {
  const double poly_b = L.quad ? 0.0 : 4.0 * (L.nf + 1) + 4.0 * L.nnz;
  return {{"scan", 8.0 * L.nv + 4},
          {L.quad ? "spgemm_symbolic_quad" : "spgemm_symbolic_poly", 8.0 * L.nnz + 8.0 * L.nv + 8.0 * L.nnz + poly_b},
          {"scan", 8.0 * L.nv + 4}};
}

StageBytes Plan::number_stage(const LevelPlan& L, bool faces) const {
  const double poly_b = L.quad ? 0.0 : 4.0 * (L.nf + 1) + 4.0 * L.nnz;
  return {faces ? (L.quad ? "number_facepoints_quad" : "number_facepoints_poly") : "number",
          12.0 * L.nv + 12.0 * L.nnz + 8.0 * L.nnz + (L.bnd ? 4.0 * (double)L.ne : 0.0) + poly_b +
              (faces ? 4.0 * L.nnz + 16.0 * L.nv + 16.0 * L.nf : 0.0)};
}

// A small mesh's first level: gather, analysis and numbering in one launch.
void Plan::record_small(LevelPlan& L, bool faces) {
  LevelView V = L.view(d_flags_, late_);
  V.ci = reinterpret_cast<int32_t*>(L.ci);
  V.bnd = L.bnd;
  V.report = report_;
  std::vector<StageBytes> stages = gather_stages(L);
  for (const StageBytes& s : analysis_stages(L)) stages.push_back(s);
  stages.push_back(number_stage(L, faces));
  // the inputs, what the gather writes, M^T's rows and offsets and the (edge,
  // twin) pairs; face points
  const double bytes = gather_bytes(L) + 16.0 * L.nnz + 4.0 * L.nv + (faces ? 16.0 * L.nv + 16.0 * L.nf : 0.0);
  ProfScope ps(st_, {L.quad ? "first_level_small_quad" : "first_level_small_poly", bytes}, std::move(stages));
  launch_first_small(L.quad, scheme_, scheme_ == kLAK, V, faces, st_);
}

void Plan::prepare() {
  for (auto& J : jobs_) {
    if (J.in.type != SLAK_TRI && J.in.type != SLAK_QUAD && J.in.type != SLAK_POLY)
      throw Error(SLAK_ERR_INVALID_ARGUMENT, "unknown mesh type");
    if (J.target < 0 || J.target > 12) throw Error(SLAK_ERR_INVALID_ARGUMENT, "target level out of range");
    J.levels = J.in.type != SLAK_QUAD ? std::max(1, J.target) : J.target;
    if (J.levels <= 0) continue;
    if (!J.in.ids || !J.in.verts) throw Error(SLAK_ERR_INVALID_ARGUMENT, "mesh ids/verts must not be null");
    if (!J.in.ptr) {
      if (J.in.type == SLAK_POLY) throw Error(SLAK_ERR_INVALID_ARGUMENT, "POLY mesh without ptr");
      int k = J.in.type == SLAK_QUAD ? 4 : 3;
      if ((int64_t)J.in.nnz != k * (int64_t)J.in.nfaces)
        throw Error(SLAK_ERR_INVALID_ARGUMENT, "nnz != face order * nfaces");
    }
    check_i32((int64_t)J.in.nverts, "nverts");
    check_i32((int64_t)J.in.nfaces, "nfaces");
    check_i32((int64_t)J.in.nnz, "nnz");
  }
  bool any = false;
  for (auto& J : jobs_) any |= J.levels > 0;
  if (!any) {
    prepared_ = true;
    return;
  }
  plan_first_level();
  LevelPlan& L1 = levels_[0];
  const int nseg = (int)L1.segs.size();
  // a single mesh numbers its edges before the read-back: the first upload
  // gives it nnz >= ne as the edge-id bound and a flag buffer of that size
  const bool early = nseg == 1 && jobs_.size() == 1;
  early_p1_ = nullptr;
  early_faces_ = false;
  if (early) {
    L1.segs[0].ne = L1.segs[0].nnz;
    L1.bnd = arena_.get_n<int32_t>(L1.nnz);
    // when the first level feeds another, its positions go to a plan buffer
    // (sized for nnz >= ne edge points) and the early numbering also forms
    // the face points
    const MeshJob& J = jobs_[L1.jobs[0]];
    if (J.levels >= 2) {
      early_p1_cap_ = (int64_t)J.in.nverts + (int64_t)J.in.nfaces + (int64_t)J.in.nnz + 8;  // + line padding
      early_p1_ = arena_.get_n<float4>(early_p1_cap_);
      L1.segs[0].dst_verts = early_p1_;
    }
  }
  if (!host_words_.p) host_words_.p = pinned_acquire((size_t)(kReportAt + 2 + kRowHistBins + nseg + 1) * 4, host_words_.cap);
  late_ = reinterpret_cast<int32_t*>(host_words_.p);
  report_ = late_ + kReportAt;
  *late_ = 0;
  *report_ = 0;
  // a small mesh's first level is one launch, which zeroes what it needs
  const bool small = early && first_level_is_small(L1.view(nullptr, nullptr));
  upload_tables(0, 1, staging_first_, !small);

  // 1. validate + gather (the state block is zeroed with the table upload)
  if (!small) {
    record_gather(L1);
    if (P1_) launch_gather_verts(L1.table(), (int32_t)L1.nv, P1_, st_);
  }
  auto fail_if = [&](int fl) {
    if (!fl) return;
    std::vector<int> mf(nseg, 0);
    // the report may have come from a launch that is still running (a small
    // mesh's), and the copy does not wait for a non-blocking stream
    SLAK_HIP_CHECK(hipStreamSynchronize(st_));
    SLAK_HIP_CHECK(hipMemcpy(mf.data(), L1.d_mflags, nseg * sizeof(int), hipMemcpyDeviceToHost));
    for (int k = 0; k < nseg; ++k) jobs_[L1.jobs[k]].bad_flags = mf[k];
    throw Error(SLAK_ERR_INVALID_MESH, describe_failure(fl));
  };
  // 2. first-level analysis: M^T, owned-edge counts, per-mesh edge totals
  // (its kernels do nothing on an input the gather flagged; the flags come
  // back with the edge counts in one round trip)
  if (small)
    record_small(L1, early_p1_ != nullptr);
  else
    record_analysis(L1);
  std::vector<int64_t> hb(kRowHistBins + nseg + 1, 0);
  // a single mesh numbers its edges (and forms its face points) meanwhile (a
  // small one in that one launch)
  if (early) {
    if (!small) launch_number(L1, early_p1_ != nullptr, true);
  } else {
    LevelView V = L1.view(d_flags_, late_);
    V.hist_rows = d_state_ + kStateRowHist;
    V.bounds = d_state_ + kStateBounds;
    V.report = report_;
    V.ngroups = (int32_t)n_groups_;
    launch_report(V, st_);
  }
  wait_report();
  fail_if(report_[1]);
  for (int b = 0; b < kRowHistBins; ++b) hb[b] = report_[2 + b];
  for (int k = 0; k <= nseg; ++k) hb[kRowHistBins + k] = report_[2 + kRowHistBins + k];
  // the early numbering was recorded before its edge count was known: its
  // boundary-flag writes (4 bytes per edge) join its algorithmic bytes now
  if (early && Profiler::get().enabled())
    Profiler::get().amend_last(L1.quad ? "number_facepoints_quad" : "number_facepoints_poly",
                               4.0 * (double)hb[kRowHistBins + 1]);
  number_early_ = early;
  early_faces_ = early && early_p1_ != nullptr;
  const int64_t* bounds = hb.data() + kRowHistBins;
  // 3. closed-form sizes of every later level
  int Lmax = 0;
  for (int k = 0; k < nseg; ++k) {
    MeshJob& J = jobs_[L1.jobs[k]];
    int lv = J.levels;
    Lmax = std::max(Lmax, lv);
    J.nv.assign(lv + 1, 0);
    J.nf.assign(lv + 1, 0);
    J.nnz.assign(lv + 1, 0);
    J.ne.assign(lv + 1, 0);
    J.nv[0] = (int64_t)J.in.nverts;
    J.nf[0] = (int64_t)J.in.nfaces;
    J.nnz[0] = (int64_t)J.in.nnz;
    J.ne[0] = bounds[k + 1] - bounds[k];
    int64_t next = 2 * J.ne[0] - J.nnz[0];  // boundary edges
    if (next < 0) throw Error(SLAK_ERR_INTERNAL, "inconsistent edge count");
    for (int l = 1; l <= lv; ++l) {
      J.nv[l] = J.nv[l - 1] + J.nf[l - 1] + J.ne[l - 1];
      J.nf[l] = J.nnz[l - 1];
      J.nnz[l] = 4 * J.nnz[l - 1];
      int64_t nx = next << l;
      J.ne[l] = (J.nnz[l] - nx) / 2 + nx;
      check_i32(J.nv[l], "refined vertices");
      check_i32(J.nnz[l], "refined corners");
    }
  }

  // 4. level unions, destinations and outputs
  const bool lak_scheme = scheme_ == kLAK;
  auto out_alloc = [&](size_t bytes) -> void* {
    if (mode_ == OutputMode::kSeparate) return pool().alloc(bytes);
    return nullptr;  // carved from pooled blocks below
  };
  // pooled outputs: one block per kind
  // each mesh's pooled arrays start on a 128-byte line: the int4 and 64-byte
  // stores of the final kernels then never straddle lines (a pointer array
  // of nf + 1 ints would otherwise shift every later mesh by 4 bytes)
  auto line_v = [](int64_t n) { return (n + 7) & ~(int64_t)7; };     // float4
  auto line_i = [](int64_t n) { return (n + 31) & ~(int64_t)31; };   // int32
  int64_t tot_v = 0, tot_i = 0, tot_p = 0;
  for (auto& J : jobs_)
    if (J.levels > 0) {
      tot_v += line_v(J.nv[J.levels]);
      tot_i += line_i(4 * J.nnz[J.levels - 1]);
      tot_p += line_i(J.nf[J.levels] + 1);
    }
  float4* pool_v = nullptr;
  int32_t *pool_i = nullptr, *pool_p = nullptr, *pool_a = nullptr;
  if (mode_ == OutputMode::kPooled) {
    pool_v = arena_.get_n<float4>(tot_v);
    pool_i = arena_.get_n<int32_t>(tot_i);
    if (lak_scheme) {
      pool_p = arena_.get_n<int32_t>(tot_p);
      pool_a = arena_.get_n<int32_t>(tot_i);
    }
  }
  int64_t ov = 0, oi = 0, op = 0;
  for (auto& J : jobs_) {
    if (J.levels <= 0) continue;
    int64_t nvo = J.nv[J.levels], nio = 4 * J.nnz[J.levels - 1], npo = J.nf[J.levels] + 1;
    const bool lak_form = lak_scheme && J.lak_form;
    if (mode_ == OutputMode::kSeparate) {
      J.out_verts = static_cast<float4*>(out_alloc(nvo * sizeof(float4)));
      J.out_ids = static_cast<int32_t*>(out_alloc(nio * sizeof(int32_t)));
      if (lak_form) {
        J.out_ptr = static_cast<int32_t*>(out_alloc(npo * sizeof(int32_t)));
        J.out_vals = static_cast<int32_t*>(out_alloc(nio * sizeof(int32_t)));
      }
    } else {
      J.out_verts = pool_v + ov;
      J.out_ids = pool_i + oi;
      if (lak_form) {
        J.out_ptr = pool_p + op;
        J.out_vals = pool_a + oi;
      }
    }
    ov += line_v(nvo);
    oi += line_i(nio);
    op += line_i(npo);
  }

  {
    const char* e = std::getenv("SLAK_FINAL_TABLE");  // one mesh through the table path too
    force_final_table_ = e && std::atoi(e) != 0;
  }
  // k_final computes the last level of every mesh refined two or more levels
  {
    const char* e = std::getenv("SLAK_FUSED_FINAL");
    const bool allow = !e || std::atoi(e) != 0;
    // k_final_deep: closed LAK meshes whose mesh three levels back is a
    // refined one (it gathers a third of what k_final does, and the level
    // before the last two writes no structure)
    const char* d = std::getenv("SLAK_FINAL_DEEP");
    const char* q = std::getenv("SLAK_FUSED_POS");
    const bool allow_deep = allow && scheme_ == kLAK && (!d || std::atoi(d) != 0) && (!q || std::atoi(q) != 0);
    for (int j : levels_[0].jobs) {
      MeshJob& J = jobs_[j];
      J.fused = allow && J.levels >= 2;
      J.deep = allow_deep && J.levels >= 4 && J.nnz[0] > 0 && 2 * J.ne[0] == J.nnz[0];  // (no faces: no edge owners)
      J.p1 = nullptr;
      J.p2 = nullptr;
      J.own_base = -1;
      if (J.nnz[0] == 0) faceless_.push_back(j);
    }
    // Two levels of thousands of tiny polygon meshes: k_final's blocks hold one
    // mesh each, so theirs are mostly idle, and the level-by-level items of
    // their union are denser. Replays, k_final against level by level: 4096
    // meshes of 12, 54 and 96 corners 114 / 99, 154 / 137, 169 / 153 us, of 150
    // corners 187 / 187; 16384: 212 / 128 ... 449 / 538; 1024: 94 / 93 ... 125 /
    // 130. Where larger meshes hold most of the corners they stay: level-by-level
    // items at the second level would take the others' positions with them.
    if (!levels_[0].quad) {
      constexpr int64_t kTinyCorners = kBlockItems / 2, kTinyMeshes = 3072;
      auto tiny = [&](const MeshJob& J) { return J.levels == 2 && J.nnz[0] <= kTinyCorners; };
      int64_t meshes = 0, corners = 0, others = 0;
      for (int j : levels_[0].jobs) {
        const MeshJob& J = jobs_[j];
        if (tiny(J)) {
          ++meshes;
          corners += J.nnz[0];
        } else if (J.levels >= 2) {
          others += J.nnz[0];
        }
      }
      if (meshes >= kTinyMeshes && corners >= others)
        for (int j : levels_[0].jobs)
          if (tiny(jobs_[j])) jobs_[j].fused = false;
    }
  }
  // whether level l of a mesh hands on its positions alone
  auto positions_only = [](const MeshJob& J, int l) {
    return (J.fused && J.levels == l + 1) || (J.deep && J.levels == l + 2);
  };
  // one arena block for the level buffers that follow (positions and ids
  // handed on, the positions for k_final, the alternating structure, the
  // boundary flags and their scan, the tables), from the closed-form sizes
  // of what the level loop below allocates; anything beyond it comes from
  // the pool as before
  {
    auto line = [](int64_t n, size_t elem) { return ((size_t)std::max<int64_t>(n, 1) * elem + 255) & ~(size_t)255; };
    size_t est = 0;
    int64_t mnv = 0, mnnz = 0, mne = 0;
    for (int l = 1; l <= Lmax; ++l) {
      int64_t nv = 0, pad = 0, ids = 0, snv = 0, snnz = 0, ne = 0;
      for (int j : levels_[0].jobs) {
        const MeshJob& J = jobs_[j];
        const bool to_final = positions_only(J, l);
        if (J.levels > l) {  // positions handed on (to the union or to k_final)
          nv += J.nv[l];
          pad += 8;
          if (!to_final) ids += J.nnz[l];
        }
        if (J.levels > l && !to_final) {  // index l's structure: level l + 1 runs it
          snv += J.nv[l];
          snnz += J.nnz[l];
        }
        if (J.levels >= l) ne += J.ne[l - 1];
      }
      est += line(nv + pad, 16) + 256 + line(ids, 4);
      mnv = std::max(mnv, snv);
      mnnz = std::max(mnnz, snnz);
      mne = std::max(mne, ne);
    }
    est += 2 * (line(mnv + 1, 4) + 2 * line(mnnz, 8) + line(mnnz, 4));
    est += (lak_scheme ? 4 : 2) * line(mne + 1, 4) + line(scan_partials_len(mne), 8);
    est += (size_t)1 << 20;
    if (Lmax >= 1) arena_.reserve(est);
  }
  // level l (1-based) consumes sizes index l-1 and produces index l
  int64_t max_nv = 0, max_nnz = 0;
  levels_.resize(Lmax);
  for (int l = 1; l <= Lmax; ++l) {
    LevelPlan& L = levels_[l - 1];
    if (l > 1) {
      LevelPlan& prev = levels_[l - 2];
      L.quad = true;
      L.jobs.clear();
      L.segs.clear();
      L.vbase.clear();
      L.fbase.clear();
      L.cbase.clear();
      int64_t vb = 0, fb = 0, cb = 0, eb = 0;
      L.fin = FinalTable{};
      L.pos = FinalTable{};
      L.deep = FinalTable{};
      L.pos_fused = false;
      for (int j : prev.jobs) {
        MeshJob& J = jobs_[j];
        if (J.levels < l) continue;
        if (J.fused && J.levels == l) {  // formed by k_final, outside the union
          L.fin.jobs.push_back(j);
          continue;
        }
        if (J.deep && J.levels == l + 1) {  // positions here, then the output, both outside the union
          L.deep.jobs.push_back(j);
          continue;
        }
        SegDesc S{};
        S.vb = vb;
        S.fb = fb;
        S.cb = cb;
        S.eb = eb;
        S.nv = (int32_t)J.nv[l - 1];
        S.nf = (int32_t)J.nf[l - 1];
        S.nnz = J.nnz[l - 1];
        L.jobs.push_back(j);
        L.segs.push_back(S);
        L.vbase.push_back(vb);
        L.fbase.push_back(fb);
        L.cbase.push_back(cb);
        vb += S.nv;
        fb += S.nf;
        cb += S.nnz;
        eb += J.ne[l - 1];
      }
      L.vbase.push_back(vb);
      L.fbase.push_back(fb);
      L.cbase.push_back(cb);
      L.nv = vb;
      L.nf = fb;
      L.nnz = cb;
      L.ne = eb;
      check_i32(L.nv, "union vertices of level " + std::to_string(l));
      check_i32(L.nnz, "union corners of level " + std::to_string(l));
      max_nv = std::max(max_nv, L.nv);
      max_nnz = std::max(max_nnz, L.nnz);
    }
    // destinations of this level's segments; a mesh whose next level is its
    // fused last one hands on its positions only, outside the next union
    auto to_final = [&](const MeshJob& J) { return positions_only(J, l); };
    int64_t nv_next = 0, nnz_next = 0;
    for (int j : L.jobs)
      if (jobs_[j].levels > l && !to_final(jobs_[j])) {
        nv_next += jobs_[j].nv[l];
        nnz_next += jobs_[j].nnz[l];
      }
    int64_t p1_total = 0, p1_off = 0;  // one block for the positions handed to k_final
    for (int j : L.jobs)
      if (to_final(jobs_[j])) p1_total += (jobs_[j].nv[l] + 7) & ~(int64_t)7;
    for (int j : L.deep.jobs) p1_total += (jobs_[j].nv[l] + 7) & ~(int64_t)7;
    // the first level's positions of a single mesh: the buffer the early
    // numbering has written the face points into
    float4* early = l == 1 && early_faces_ && nv_next + p1_total <= early_p1_cap_ ? early_p1_ : nullptr;
    if (l == 1 && early_faces_ && !early) throw Error(SLAK_ERR_INTERNAL, "first-level positions exceed their buffer");
    float4* Un_P = nv_next ? (early ? early : arena_.get_n<float4>(nv_next)) : nullptr;
    int32_t* Un_ids = nnz_next ? arena_.get_n<int32_t>(nnz_next) : nullptr;
    float4* p1_block = p1_total ? (early ? early : arena_.get_n<float4>(p1_total)) : nullptr;
    int64_t vbn = 0, cbn = 0, ebn = 0, own = 0;
    for (size_t k = 0; k < L.segs.size(); ++k) {
      MeshJob& J = jobs_[L.jobs[k]];
      SegDesc& S = L.segs[k];
      S.ne = J.ne[l - 1];
      S.next_own = -1;
      if (l == 1) S.eb = bounds[k];
      L.boundary |= 2 * J.ne[l - 1] != J.nnz[l - 1];  // n_ext = 2 n_e - nnz
      if (J.levels == l) {
        S.dst_verts = J.out_verts;
        S.dst_ids = J.out_ids;
        S.dst_ptr = J.out_ptr;
        S.dst_vals = J.out_vals;
        S.id_offset = 0;
        S.next_vb = -1;
        S.next_cb = -1;
        S.next_eb = -1;
        S.dst_final = 1;
      } else if (to_final(J)) {
        S.dst_verts = p1_block + p1_off;
        p1_off += (J.nv[l] + 7) & ~(int64_t)7;  // 128-byte lines
        (J.levels == l + 1 ? J.p1 : J.p2) = S.dst_verts;
        S.dst_ids = nullptr;
        S.dst_ptr = nullptr;
        S.dst_vals = nullptr;
        S.id_offset = 0;
        S.next_vb = -1;
        S.next_cb = -1;
        S.next_eb = -1;
      } else {
        S.dst_verts = Un_P + vbn;
        S.dst_ids = Un_ids ? Un_ids + cbn : nullptr;
        S.dst_ptr = nullptr;
        S.dst_vals = nullptr;
        S.id_offset = vbn;
        S.next_vb = vbn;
        S.next_cb = cbn;
        S.next_eb = ebn;
        vbn += J.nv[l];
        cbn += J.nnz[l];
        ebn += J.ne[l];
        if (J.deep && J.levels == l + 3) {  // a multiple of 4 edges: closed refined meshes only
          S.next_own = J.own_base = own;
          own += J.ne[l];
        }
      }
    }
    for (int j : L.deep.jobs) {
      jobs_[j].p1 = p1_block + p1_off;
      p1_off += (jobs_[j].nv[l] + 7) & ~(int64_t)7;
    }
    if (own > 0) levels_[l].own = arena_.get_n<int2>(own);
    if (l == 1) L.ne = bounds[nseg];
    L.next_nv = nv_next;
    L.next_nnz = nnz_next;
    if (l < Lmax) {
      LevelPlan& nx = levels_[l];
      nx.ids = Un_ids;
      nx.P = Un_P;
    }
  }
  // Levels >= 2 receive their structure from the level before (two
  // alternating buffers of each kind, sized for the largest level); the
  // boundary flags and their scan are one buffer pair shared by every level.
  // Only the last level's union can be empty (every mesh in it fused), and
  // then nothing is written for it.
  int Lstruct = Lmax;  // last level whose input structure is written
  while (Lstruct >= 2 && levels_[Lstruct - 1].segs.empty()) --Lstruct;
  if (Lstruct >= 2) {
    int32_t* mt_ptr[2] = {arena_.get_n<int32_t>(max_nv + 1),
                          Lstruct >= 3 ? arena_.get_n<int32_t>(max_nv + 1) : nullptr};
    int2* mt_row[2] = {arena_.get_n<int2>(max_nnz), Lstruct >= 3 ? arena_.get_n<int2>(max_nnz) : nullptr};
    int2* mt_ci[2] = {arena_.get_n<int2>(max_nnz), Lstruct >= 3 ? arena_.get_n<int2>(max_nnz) : nullptr};
    int32_t* mt_pos[2] = {nullptr, nullptr};
    if (scheme_ == kSLAK) {
      mt_pos[0] = arena_.get_n<int32_t>(max_nnz);
      if (Lstruct >= 3) mt_pos[1] = arena_.get_n<int32_t>(max_nnz);
    }
    for (int l = 2; l <= Lstruct; ++l) {
      LevelPlan& L = levels_[l - 1];
      L.tptr = mt_ptr[l % 2];
      L.trow = mt_row[l % 2];
      L.ci = mt_ci[l % 2];
      L.mpos = mt_pos[l % 2];
      levels_[l - 2].ntptr = L.tptr;
      levels_[l - 2].ntrow = L.trow;
      levels_[l - 2].nci = L.ci;
      levels_[l - 2].nmpos = L.mpos;
    }
  }
  int64_t max_ne = 0;
  for (int l = 1; l <= Lstruct; ++l)
    if (levels_[l - 1].boundary) max_ne = std::max(max_ne, levels_[l - 1].ne);
  if (max_ne > 0) {
    int32_t* bnd = arena_.get_n<int32_t>(max_ne);
    int32_t* blk = arena_.get_n<int32_t>(max_ne + 1);
    // LAK: later levels receive their ranks from the level before, which reads
    // its own meanwhile (two alternating buffers)
    int32_t* ranks[2] = {nullptr, nullptr};
    if (lak_scheme && Lstruct >= 2) ranks[0] = arena_.get_n<int32_t>(max_ne + 1);
    if (lak_scheme && Lstruct >= 3) ranks[1] = arena_.get_n<int32_t>(max_ne + 1);
    for (int l = 1; l <= Lstruct; ++l) {
      LevelPlan& L = levels_[l - 1];
      if (!L.boundary) continue;
      if (lak_scheme && l >= 2) {
        L.blk = ranks[l % 2];
        levels_[l - 2].nbnd = L.blk;
        continue;
      }
      if (!(l == 1 && number_early_)) L.bnd = bnd;  // the early numbering wrote level 1's own
      L.blk = blk;
      if (l >= 2) levels_[l - 2].nbnd = bnd;
    }
    int64_t need2 = scan_partials_len(max_ne);
    if (need2 > partial_len_) {
      d_partial_ = arena_.get_n<int64_t>(need2);
      partial_len_ = need2;
    }
  }
  // the first level's rows per block, now with the row-length spread (the
  // numbering after the read-back and every graph replay use it)
  {
    const RowTiling rt = autotune_rows(levels_[0].nv, levels_[0].nnz, hb.data());
    levels_[0].rows = rt.rows;
    levels_[0].tile = rt.tile;
  }
  // k_final tables: per fused mesh, its segment of M (the level before's
  // union), the positions of M1 and its outputs
  std::vector<int> seg_in_m(jobs_.size(), -1);  // job -> its segment of M
  const char* pe = std::getenv("SLAK_FUSED_POS");
  const bool allow_pos = !pe || std::atoi(pe) != 0;
  lak_ = LakTable{};
  for (int l = 2; l <= Lmax; ++l) {
    LevelPlan& L = levels_[l - 1];
    const LevelPlan& M = levels_[l - 2];
    for (size_t k = 0; k < M.jobs.size(); ++k) seg_in_m[M.jobs[k]] = (int)k;
    auto segment = [&](int j, const float4* P) -> const SegDesc& {
      if (seg_in_m[j] < 0 || !P) throw Error(SLAK_ERR_INTERNAL, "fused level without its input");
      return M.segs[seg_in_m[j]];
    };
    L.fin.segs.reserve(L.fin.jobs.size());
    L.deep.segs.reserve(L.deep.jobs.size());
    // meshes whose last level is l
    for (int j : L.fin.jobs) add_final_seg(L.fin, l, j, segment(j, jobs_[j].p1), jobs_[j].p1, jobs_[j].out_verts);
    plan_blocks(L.fin, M.quad, false);
    // a level whose every segment hands on its positions alone: its positions
    // from the structure two levels back too
    bool pos = allow_pos && !L.segs.empty();
    for (int j : L.jobs) pos = pos && positions_only(jobs_[j], l);
    L.pos.segs.reserve((pos ? L.jobs.size() : 0) + L.deep.jobs.size());
    if (pos) {
      L.pos_fused = true;
      for (size_t k = 0; k < L.segs.size(); ++k) {
        const int j = L.jobs[k];
        const float4* P = L.P + L.segs[k].vb;
        L.pos.jobs.push_back(j);
        add_final_seg(L.pos, l, j, segment(j, P), P, L.segs[k].dst_verts);
      }
    }
    // meshes whose last level is l + 1, from the mesh two levels before l
    for (int j : L.deep.jobs) {
      MeshJob& J = jobs_[j];
      L.pos.jobs.push_back(j);
      add_final_seg(L.pos, l, j, segment(j, J.p2), J.p2, J.p1);
      add_final_seg(L.deep, l, j, segment(j, J.p1), J.p1, J.out_verts);
      if (J.own_base < 0) throw Error(SLAK_ERR_INTERNAL, "deep final level without its edge owners");
      L.deep.segs.back().m.eb = J.own_base;
    }
    plan_blocks(L.pos, M.quad, false);
    plan_blocks(L.deep, M.quad, true);
  }
  // a level whose meshes all come from k_final runs no refine or vertex
  // items over its structure: only k_final reads its M^T rows, and it needs
  // their corners alone
  for (size_t i = 1; i < levels_.size(); ++i)
    levels_[i].rows_x = levels_[i].segs.empty() || levels_[i].pos_fused;
  upload_tables(0, (int)levels_.size(), staging_all_);
  prepared_ = true;
}

// The first level's edge numbering (E of the mapped SpGEMM: edge id and twin
// of every half-edge, boundary flags), with its face points in the same
// launch when faces is set.
void Plan::launch_number(LevelPlan& L, bool faces, bool rep) {
  LevelView V = L.view(d_flags_, late_);
  V.ci = reinterpret_cast<int32_t*>(L.ci);
  V.bnd = L.bnd;
  V.planned = replayed_ ? 1 : 0;
  if (rep) {
    V.report = report_;
    V.hist_rows = d_state_ + kStateRowHist;
    V.ngroups = (int32_t)n_groups_;
  }
  const StageBytes stage = number_stage(L, faces);
  ProfScope ps(st_, stage.name, stage.bytes);
  launch_number_faces(L.quad, scheme_, V, faces, st_);
}

// Vertex runs of the mesh two levels before job J's level l (the mesh M of its
// k_final): the original vertices, then the face points and edge points of
// every level before M (the leading classes as one past kMaxVSeg); one run if
// the sizes do not add up. more: items that follow, a run of their own.
static void set_runs(VertexRuns& R, const MeshJob& J, int l, int32_t more = 0) {
  const int levels = std::max(l - 2, 0), classes = 1 + 2 * levels + (more ? 1 : 0);
  int skip = std::max(classes - kMaxVSeg, 0);
  int64_t end = 0;
  R.n = 0;
  R.first[0] = 0;
  auto add = [&](int64_t c) {
    end += c;
    if (skip > 0)
      --skip;
    else
      R.first[++R.n] = (int32_t)end;
  };
  add(J.nv[0]);
  for (int k = 0; k < levels; ++k) {
    add(J.nf[k]);
    add(J.ne[k]);
  }
  if (end != J.nv[levels]) {
    skip = 0;
    R.n = 0;
    end = 0;
    add(J.nv[levels]);
  }
  if (more) add(more);
}

// The blocks of a table's meshes, mesh by mesh, and (several meshes) the mesh
// of every block.
void Plan::plan_blocks(FinalTable& T, bool quad, bool deep) {
  int64_t blocks = 0;
  const bool table = final_table(T);
  if (table) T.block_seg.reserve(2 * T.segs.size());  // (a corner and a vertex block of each mesh at least)
  for (size_t k = 0; k < T.segs.size(); ++k) {
    FinalSeg& F = T.segs[k];
    F.block0 = (int32_t)blocks;
    blocks += plan_final_blocks(F, quad, deep);
    check_i32(blocks * kBlockItems / 2, "items of a final level");
    if (!table) continue;
    T.block_seg.resize((size_t)blocks, (int32_t)k);
    if (!F.m.out_vals) continue;
    LakSeg A{};
    A.block0 = (int32_t)lak_.block_seg.size();
    A.n = (deep ? 4 : 1) * F.m.nnz;
    A.vals = F.m.out_vals;
    A.ptr = F.m.out_ptr;
    const int64_t lak = (int64_t)A.block0 + ((int64_t)A.n + kBlockItems - 1) / kBlockItems;
    check_i32(lak * kBlockItems / 2, "items of the LAK form");
    lak_.block_seg.resize((size_t)lak, (int32_t)lak_.segs.size());
    lak_.segs.push_back(A);
    lak_.bytes += 4.0 * (A.ptr ? 4.0 * A.n + 1 : 0.0) + 64.0 * A.n;
  }
}

// the meshes of a table as a launch's arguments
void Plan::set_final_table(FinalView& V, const FinalTable& T) const {
  if (!final_table(T)) {
    V.one = T.segs[0];
    return;
  }
  V.segs = T.d_segs;
  V.block_seg = T.d_block_seg;
  V.nblocks = (int32_t)T.block_seg.size();
}

// One mesh of a k_final table: m is its segment of M (of N for k_final_deep),
// P1 the positions of M1. The output level also writes the job's quads and
// LAK form; other levels positions alone.
void Plan::add_final_seg(FinalTable& T, int l, int job, const SegDesc& m, const float4* P1, float4* positions) {
  const MeshJob& J = jobs_[job];
  FinalSeg F{};
  F.m.cb = m.cb;
  F.m.vb = m.vb;
  F.m.eb = m.eb;
  F.m.fb = m.fb;
  F.m.nv = m.nv;
  F.m.nf = m.nf;
  F.m.ne = (int32_t)m.ne;
  F.m.nnz = (int32_t)m.nnz;
  F.m.P1 = P1;
  F.m.out_verts = positions;
  if (positions == J.out_verts) {
    F.m.out_ids = J.out_ids;
    F.m.out_ptr = J.out_ptr;
    F.m.out_vals = J.out_vals;
  }
  set_runs(F.runs, J, l, levels_[l - 2].quad ? 0 : m.nf);  // (polygons' face points have items of their own)
  T.segs.push_back(F);
}

// Output positions above which a launch's edge points bypass the caches: 7/8
// of the 256 MB last-level cache (measured between 201 MB, where it costs 4 %,
// and 268 MB, where it gives 7 % (k_final_deep) and 13 % (k_final)).
constexpr double kStreamBytes = 224.0 * (1 << 20);

// k_final_deep over the meshes of table T, whose last level is l + 1, from the
// structure of their mesh two levels before l (level l - 1's union) and their
// positions of level l: launched right after those positions, before anything
// of level l overwrites the structure.
void Plan::launch_deep(int l, FinalTable& T) {
  const LevelPlan& N = levels_[l - 2];
  FinalView V{};
  V.ids = N.ids;
  V.ci = N.ci;
  V.tptr = N.tptr;
  V.trow = N.trow;
  V.trow_x = N.rows_x ? reinterpret_cast<const int32_t*>(N.trow) : nullptr;
  V.own = N.own;
  V.stop = stop();
  set_final_table(V, T);
  const bool multi = final_table(T);
  // algorithmic bytes: reads N's ids, (edge, twin) pairs, edge owners, M^T
  // rows and offsets and the positions of M1; writes the output positions and
  // quads (and one mesh's LAK form)
  double bytes = 0, positions = 0;
  for (int j : T.jobs) {
    const MeshJob& J = jobs_[j];
    const double nnz = (double)J.nnz[l - 2], nnz1 = (double)J.nnz[l];
    bytes += 12.0 * nnz + 8.0 * (double)J.ne[l - 2] + (N.rows_x ? 4.0 : 8.0) * nnz + 4.0 * (double)J.nv[l - 2] +
             16.0 * (double)J.nv[l] + 16.0 * ((double)J.nv[l] + (double)J.nf[l] + (double)J.ne[l]) + 16.0 * nnz1;
    if (J.out_ptr && !multi) bytes += 4.0 * (nnz1 + 1) + 16.0 * nnz1;
    positions += 16.0 * ((double)J.nv[l] + (double)J.nf[l] + (double)J.ne[l]);
  }
  V.stream = positions > kStreamBytes;
  {
    ProfScope ps(st_, "refine_vertex_final_quad", bytes);
    launch_final_deep(V, st_);
  }
}

// k_final over the meshes of table T at level l, from the structure of their
// mesh two levels back (the previous level's union): launched before anything
// of level l overwrites that structure (the boundary scan buffer, the
// alternating M^T buffers). ids: the output level (quads, LAK form,
// positions); otherwise positions only.
void Plan::launch_final_table(int l, FinalTable& T, bool ids, const char* stage) {
  if (T.empty()) return;
  const LevelPlan& M = levels_[l - 2];
  FinalView V{};
  V.ids = M.ids;
  V.ci = M.ci;
  if (!M.quad) {
    V.fptr = M.fptr;
    V.cface = M.cface;
  }
  V.tptr = M.tptr;
  V.trow = M.trow;
  V.trow_x = M.rows_x ? reinterpret_cast<const int32_t*>(M.trow) : nullptr;
  V.blk = M.blk;
  V.mpos = M.mpos;
  V.stop = stop();
  set_final_table(V, T);
  // algorithmic bytes: reads the ids, (edge, twin) pairs, M^T rows and
  // offsets of M (boundary scan, SLAK positions) and the positions of M1;
  // writes every output position and, for the output level, the quads (and
  // the LAK form)
  // (several meshes: the LAK form is written by a launch of its own)
  const bool multi = final_table(T);
  double reads = 0, writes = 0, positions = 0;
  for (int j : T.jobs) {
    const MeshJob& J = jobs_[j];
    const double mnnz = (double)J.nnz[l - 2], mnv = (double)J.nv[l - 2], mne = (double)J.ne[l - 2];
    const double nnz1 = (double)J.nnz[l - 1], nv1 = (double)J.nv[l - 1], nf1 = (double)J.nf[l - 1];
    const double ne1 = (double)J.ne[l - 1];
    reads += (M.rows_x ? 16.0 : 20.0) * mnnz + (M.quad ? 0.0 : 4.0 * mnnz + 4.0 * ((double)J.nf[l - 2] + 1)) + 4.0 * mnv + (M.blk ? 4.0 * mne : 0.0) + (scheme_ == kSLAK ? 4.0 * mnnz : 0.0) + 16.0 * nv1;
    writes += 16.0 * nv1 + 16.0 * nf1 + 16.0 * ne1;
    positions += 16.0 * (nv1 + nf1 + ne1);
    if (ids) {
      writes += 16.0 * nnz1;
      if (J.out_ptr && !multi) writes += 4.0 * (nnz1 + 1) + 16.0 * nnz1;
    }
  }
  V.stream = ids && positions > kStreamBytes;
  {
    ProfScope ps(st_, stage, reads + writes);
    launch_final(scheme_, V, ids, st_);
  }
}

void Plan::record_level(int l) {
  LevelPlan& L = levels_[l - 1];
  if (l > 1) {
    const bool quad = levels_[l - 2].quad;
    launch_final_table(l, L.fin, true, quad ? "refine_vertex_final_quad" : "refine_vertex_final_poly");
    launch_final_table(l, L.pos, false, quad ? "refine_vertex_pos_quad" : "refine_vertex_pos_poly");
    if (!L.deep.empty()) launch_deep(l, L.deep);
  }
  if (L.segs.empty()) return;  // every mesh of the level was fused
  const double poly_b = L.quad ? 0.0 : 4.0 * (L.nf + 1) + 4.0 * L.nnz;
  const double ne = (double)L.ne;
  if (l == 1 && !number_early_) {
    // edge numbering of the first level (later levels get theirs in closed form)
    launch_number(L, true);
  }
  if (l == 1 && number_early_ && !early_faces_) {
    ProfScope ps(st_, L.quad ? "facepoints_quad" : "facepoints_poly",
                 4.0 * L.nnz + 16.0 * L.nv + 16.0 * L.nf + (L.quad ? 0.0 : 4.0 * (L.nf + 1)));
    launch_faces(L.quad, L.ids, L.fptr, L.P, (int32_t)L.nf, L.table(), stop(), st_);
  }
  if (L.blk && (l == 1 || scheme_ == kSLAK)) {
    ProfScope ps(st_, "scan", 8.0 * ne + 4);
    launch_scan(L.bnd, L.blk, L.ne, d_partial_, late_, st_);
  }
  if (L.pos_fused) return;  // its positions came from k_final; the scan above serves the next level's
  if (l > 1) {
    ProfScope ps(st_, L.quad ? "facepoints_quad" : "facepoints_poly",
                 4.0 * L.nnz + 16.0 * L.nv + 16.0 * L.nf + (L.quad ? 0.0 : 4.0 * (L.nf + 1)));
    launch_faces(L.quad, L.ids, L.fptr, L.P, (int32_t)L.nf, L.table(), stop(), st_);
  }
  RefineView R{};
  R.ids = L.ids;
  R.fptr = L.fptr;
  R.cface = L.cface;
  R.P = L.P;
  R.nv = (int32_t)L.nv;
  R.nf = (int32_t)L.nf;
  R.nnz = L.nnz;
  R.tptr = L.tptr;
  R.trow = L.trow;
  R.ci = L.ci;
  R.blk = L.blk;
  R.mpos = L.mpos;
  R.seg = L.table();
  R.stop = stop();
  R.ntptr = L.ntptr;
  R.ntrow = L.ntrow;
  R.nci = L.nci;
  R.nbnd = L.nbnd;
  R.nmpos = L.nmpos;
  R.nown = l < (int)levels_.size() ? levels_[l].own : nullptr;
  R.next_nv = (int32_t)L.next_nv;
  R.next_nnz = (int32_t)L.next_nnz;
  R.next_rows_x = l < (int)levels_.size() && levels_[l].rows_x ? 1 : 0;
  if (L.segs.size() == 1 && l >= 2) {
    // one mesh: its vertex classes (the original vertices, then the face and
    // edge points of every earlier level) as runs in step with the corners
    set_runs(R.runs, jobs_[L.jobs[0]], l + 1);
  }
  const bool next = L.ntptr != nullptr;
  {
    // algorithmic bytes of the fused launch, each array once: reads ids,
    // (edge, twin) pairs, positions, face points and the M^T rows; writes
    // edge and vertex points, the refined quads of the meshes that keep them
    // (not those whose next level is formed by k_final) and, for the meshes
    // that feed another level, their (edge, twin) pairs, M^T rows and
    // offsets, boundary flags and (SLAK) M^T positions
    double reads = 4.0 * L.nnz + 8.0 * L.nnz + 16.0 * L.nv + 16.0 * L.nf + 4.0 * L.nv + 8.0 * L.nnz +
                   (L.blk ? 4.0 * ne : 0.0) + poly_b;
    double writes = 16.0 * ne + 16.0 * L.nv;
    for (const SegDesc& S : L.segs) {
      const double snnz = (double)S.nnz, sne = (double)S.ne;
      if (S.dst_ids) writes += 16.0 * snnz;
      if (S.dst_ptr) writes += 4.0 * (snnz + 1) + 16.0 * snnz;  // LAK form of a final level
      if (next && S.next_cb >= 0) {
        writes += (R.next_rows_x ? 48.0 : 64.0) * snnz + 4.0 * ((double)S.nv + (double)S.nf + sne) + (L.nbnd ? 4.0 * (snnz + 2.0 * sne) : 0.0) +
                  (scheme_ == kSLAK ? 16.0 * snnz : 0.0);
        if (scheme_ == kSLAK) reads += 4.0 * snnz;
        if (S.next_own >= 0) writes += 32.0 * sne;
      }
    }
    ProfScope ps(st_, L.quad ? "refine_vertex_quad" : "refine_vertex_poly", reads + writes);
    launch_level(L.quad, scheme_, R, st_);
  }
}

void Plan::launch(bool include_analysis) {
  if (levels_.empty()) return;
  replayed_ = include_analysis;
  LevelPlan& L1 = levels_[0];
  if (include_analysis) {
    number_early_ = false;  // the analysis runs again: number in order
    *late_ = 0;             // (no earlier run is in flight: finish() waits for each)
    launch_setup(nullptr, nullptr, 0, d_state_, n_state_, st_);  // a fill kernel: graph-safe
    record_gather(L1);
    if (P1_) {
      ProfScope ps(st_, "gather_verts", 32.0 * L1.nv);
      launch_gather_verts(L1.table(), (int32_t)L1.nv, P1_, st_);
    }
    record_analysis(L1);
  }
  for (int l = 1; l <= (int)levels_.size(); ++l) record_level(l);
  // the LAK form of a mesh without faces is the single offset 0, which no
  // corner item writes
  for (int j : faceless_)
    if (jobs_[j].out_ptr) launch_fill_i32(jobs_[j].out_ptr, 1, 0, st_);
  if (!lak_.segs.empty()) {
    ProfScope ps(st_, "lak_form", lak_.bytes);
    launch_lak_form(lak_.d_segs, lak_.d_block_seg, (int64_t)lak_.block_seg.size(), st_);
  }
}

void Plan::run_graph() {
  if (levels_.empty()) return;
  // The legacy default stream cannot be captured: graph plans run on a stream
  // of their own, ordered after the caller's default-stream work by an event.
  if (!capture_st_) {
    if (st_) {
      capture_st_ = st_;
    } else {
      SLAK_HIP_CHECK(hipStreamCreateWithFlags(&owned_st_, hipStreamNonBlocking));
      SLAK_HIP_CHECK(hipEventCreateWithFlags(&order_ev_, hipEventDisableTiming));
      capture_st_ = owned_st_;
    }
  }
  if (owned_st_) {
    SLAK_HIP_CHECK(hipEventRecord(order_ev_, nullptr));
    SLAK_HIP_CHECK(hipStreamWaitEvent(owned_st_, order_ev_, 0));
  }
  hipStream_t saved = st_;
  st_ = capture_st_;
  struct Restore {
    hipStream_t& ref;
    hipStream_t val;
    ~Restore() { ref = val; }
  } restore{st_, saved};
  if (!exec_) {
    // event-pair timing stays out of the captured graph
    const bool prof = Profiler::get().enabled();
    Profiler::get().set_enabled(false);
    SLAK_HIP_CHECK(hipStreamBeginCapture(st_, hipStreamCaptureModeThreadLocal));
    try {
      launch(true);
      Profiler::get().set_enabled(prof);
    } catch (...) {
      Profiler::get().set_enabled(prof);
      hipGraph_t g = nullptr;
      (void)hipStreamEndCapture(st_, &g);
      if (g) (void)hipGraphDestroy(g);
      throw;
    }
    SLAK_HIP_CHECK(hipStreamEndCapture(st_, &graph_));
    SLAK_HIP_CHECK(hipGraphInstantiate(&exec_, graph_, nullptr, nullptr, 0));
  }
  replayed_ = true;
  *late_ = 0;
  SLAK_HIP_CHECK(hipGraphLaunch(exec_, st_));
  if (owned_st_) {
    // later work on the caller's default stream sees the results
    SLAK_HIP_CHECK(hipEventRecord(order_ev_, owned_st_));
    SLAK_HIP_CHECK(hipStreamWaitEvent(nullptr, order_ev_, 0));
  }
}

void Plan::finish() {
  if (levels_.empty()) return;
  int fl = 0;
  if (replayed_) {  // the analysis ran again: its flags too
    fl = read_flags();
  } else {
    SLAK_HIP_CHECK(hipStreamSynchronize(st_));
    ++syncs_;
  }
  fl |= *late_;
  if (fl) throw Error(SLAK_ERR_INTERNAL, "refinement produced invalid topology:" + flags_message(fl));
}

void Plan::release_outputs() { outputs_released_ = true; }

size_t Plan::bytes() const { return arena_.bytes(); }

}  // namespace slak
