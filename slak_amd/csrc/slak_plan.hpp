// Multi-mesh level plans: the level chain of subdivideIteratively
// (LAKCatmullClarkImpl.cu:512-571, CatmullClarkImpl.cu:457-515) over a union
// of meshes, with every size after the first level's edge count known in
// closed form, so the whole chain can be launched back to back or captured in
// one hipGraph.
#pragma once

#include <functional>

#include <hip/hip_runtime.h>

#include <memory>
#include <string>
#include <vector>

#include "slak_c.h"
#include "slak_internal.hpp"

namespace slak {

// One caller mesh of a plan.
struct MeshJob {
  slak_mesh in{};   // caller's device mesh (never modified)
  int target = 0;   // requested level
  int levels = 0;   // levels to refine (a non-quad input gets at least one)
  bool lak_form = true;  // LAK scheme: also write ptr/vals of the final level
  // closed-form sizes of the input of level l (l = 0..levels) and its edges
  std::vector<int64_t> nv, nf, nnz, ne;
  // final outputs
  float4* out_verts = nullptr;
  int32_t* out_ids = nullptr;
  int32_t* out_ptr = nullptr;
  int32_t* out_vals = nullptr;
  int bad_flags = 0;
  // the last level is formed by k_final from the mesh two levels back;
  // p1: the positions of the level before the output (its only output)
  bool fused = false;
  float4* p1 = nullptr;
  // ... or by k_final_deep from the quad mesh three levels back (closed LAK
  // meshes of four levels or more): then the level before those two writes
  // positions only too, to p2; own_base: the mesh's edge owners
  bool deep = false;
  float4* p2 = nullptr;
  int64_t own_base = -1;
};

// Meshes whose level is formed by k_final from the structure of their mesh M
// two levels before it (k_final_deep: N, three levels before): per mesh its
// segment of M, the positions of M1, the outputs and its blocks; several
// meshes: the mesh of every block of the launch and of the LAK form's.
struct FinalTable {
  std::vector<int> jobs;
  std::vector<FinalSeg> segs;
  std::vector<int32_t> block_seg;
  FinalSeg* d_segs = nullptr;
  int32_t* d_block_seg = nullptr;
  bool empty() const { return segs.empty(); }
};

// The LAK forms of every mesh of those tables that has one, in one launch.
struct LakTable {
  std::vector<LakSeg> segs;
  std::vector<int32_t> block_seg;
  LakSeg* d_segs = nullptr;
  int32_t* d_block_seg = nullptr;
  double bytes = 0;
};

// rows per block and LDS row tile (entries) of the first level's numbering
struct RowTiling {
  int rows;
  int tile;
};

struct LevelPlan {
  bool quad = true;
  int64_t nv = 0, nf = 0, nnz = 0;  // union sizes
  const int32_t* ids = nullptr;
  const int32_t* fptr = nullptr;
  const int32_t* cface = nullptr;
  const float4* P = nullptr;
  int64_t ne = 0;           // union edges
  bool boundary = false;    // some mesh of the level has boundary edges
  int cap = kRowSlots;      // first level: M^T row length held in registers
  int rows = 256;           // first level: M^T rows per block of the numbering (autotuned)
  int tile = 1536;          // first level: its LDS row tile, entries (autotuned)
  // first-level analysis scratch (see LevelView)
  int32_t *cnt = nullptr, *slots = nullptr, *head = nullptr, *tids = nullptr, *eptr = nullptr;
  int32_t *pool = nullptr, *ecnt = nullptr;
  uint64_t *tile_sum = nullptr, *group_sum = nullptr;
  // the level's structure: M^T rows with in-neighbours, (edge id, twin) per
  // corner, boundary flags per edge and their scan (boundary levels)
  int32_t* tptr = nullptr;
  int2* trow = nullptr;
  int2* ci = nullptr;
  int32_t *bnd = nullptr, *blk = nullptr;
  int32_t* mpos = nullptr;  // M^T storage position per corner (SLAK)
  // the next level's structure, written by this level's refine and vertex kernels
  int32_t* ntptr = nullptr;
  int2* ntrow = nullptr;
  int2* nci = nullptr;
  int32_t* nbnd = nullptr;
  int32_t* nmpos = nullptr;
  int64_t next_nv = 0, next_nnz = 0;  // next level's union sizes
  std::vector<int> jobs;  // segment -> job
  std::vector<SegDesc> segs;
  std::vector<int64_t> vbase, fbase, cbase;
  // meshes whose last level is this one, formed by k_final (output quads,
  // LAK form, positions); they are not segments of this level's union
  FinalTable fin;
  // meshes whose last level is the next one, formed by k_final_deep right
  // after their positions of this level (in `pos`)
  FinalTable deep;
  int2* own = nullptr;  // edge owners of this level's meshes that k_final_deep starts from
  // every segment of this level hands its positions to k_final at the next
  // level: they are formed here by k_final's positions-only variant, and
  // this level launches no face points and no refine or vertex items
  bool pos_fused = false;
  FinalTable pos;
  // this level's M^T rows are read by k_final alone (no refine or vertex
  // items run over them): the level before writes only their corners, as
  // int32 in the row buffer
  bool rows_x = false;
  SegDesc* d_segs = nullptr;
  int64_t* d_vbase = nullptr;
  int64_t* d_fbase = nullptr;
  int64_t* d_cbase = nullptr;
  int32_t *d_vblk = nullptr, *d_fblk = nullptr, *d_cblk = nullptr;
  int* d_mflags = nullptr;
  LevelView view(int* flags, int* late) const;  // the first level's inputs and analysis arrays
  SegTable table() const {
    SegTable T{};
    T.d = d_segs;
    T.vbase = d_vbase;
    T.fbase = d_fbase;
    T.cbase = d_cbase;
    T.vblk = d_vblk;
    T.fblk = d_fblk;
    T.cblk = d_cblk;
    T.n = (int32_t)segs.size();
    T.mflags = d_mflags;
    if (T.n == 1) T.one = segs[0];
    return T;
  }
};

enum class OutputMode {
  kSeparate,  // one pool block per output array (handed to the caller)
  kPooled,    // one block per array kind for all meshes (owned by the plan)
};

class Plan {
 public:
  Plan(int scheme, std::vector<MeshJob> jobs, OutputMode mode, hipStream_t st);
  ~Plan();
  Plan(const Plan&) = delete;
  Plan& operator=(const Plan&) = delete;

  // Validates the inputs and runs the first level's analysis (one blocking
  // round trip), then sizes and allocates everything. Throws on bad input.
  void prepare();
  // Launches the chain on the plan's stream. With include_analysis the first
  // level is recomputed from the caller's meshes (used for graph replays).
  void launch(bool include_analysis);
  // Captures launch(true) into a hipGraph (once) and replays it.
  void run_graph();
  // Waits for the stream and checks the device flag word.
  void finish();
  // Hands the outputs of kSeparate plans to the caller (not freed by the plan).
  void release_outputs();

  std::vector<MeshJob>& jobs() { return jobs_; }
  LevelPlan& level(int i) { return levels_[i]; }
  int* flags() { return d_flags_; }
  int* late() { return late_; }
  Arena& arena() { return arena_; }
  int syncs() const { return syncs_; }
  hipStream_t stream() const { return st_; }
  size_t bytes() const;
  int max_levels() const { return (int)levels_.size(); }
  std::string describe_failure(int fl) const;

 private:
  void plan_first_level();
  void record_analysis(LevelPlan& L);
  void record_level(int l);
  // zero_state: also zeroes the plan's state block (first upload)
  // pinned host staging of a table upload (recycled through a process-wide
  // pool; released once the plan's stream has passed the copy)
  struct Staging {
    char* p = nullptr;
    size_t cap = 0;
  };
  void upload_tables(int l0, int l1, Staging& staging, bool zero_state = false);
  void record_gather(LevelPlan& L);
  void record_small(LevelPlan& L, bool faces);
  // algorithmic bytes of the first level's stages; of the gather's launch
  std::vector<StageBytes> gather_stages(const LevelPlan& L) const;
  double gather_bytes(const LevelPlan& L) const;
  std::vector<StageBytes> analysis_stages(const LevelPlan& L) const;
  StageBytes number_stage(const LevelPlan& L, bool faces) const;
  int read_flags();
  void wait_report();
  void launch_number(LevelPlan& L, bool faces, bool rep = false);

  int scheme_;
  std::vector<MeshJob> jobs_;
  OutputMode mode_;
  hipStream_t st_;
  Arena arena_;
  std::vector<LevelPlan> levels_;
  int* d_flags_ = nullptr;
  int64_t* d_partial_ = nullptr;
  int64_t partial_len_ = 0;
  // per-plan device state, zeroed before each run of the analysis:
  // [flags | row hist | edge bounds (nseg + 1) | mesh flags (nseg)],
  // then [pool | group sums | valence counters] (n_state_ ints in all)
  int32_t* d_state_ = nullptr;
  int64_t n_state_ = 0, n_groups_ = 0;
  Staging staging_first_, staging_all_;  // segment table uploads
  // pinned words the device writes: [late flags | pad | report] (see LevelView)
  Staging host_words_;
  int32_t* late_ = nullptr;
  int32_t* report_ = nullptr;
  bool replayed_ = false;  // the last launch ran the analysis again
  const int* stop() const { return replayed_ ? d_flags_ : nullptr; }  // see stopped()
  // first-level union gather (multi-mesh)
  float4* P1_ = nullptr;
  bool prepared_ = false;
  bool outputs_released_ = false;
  int syncs_ = 0;
  hipGraph_t graph_ = nullptr;
  hipGraphExec_t exec_ = nullptr;
  hipStream_t capture_st_ = nullptr;  // stream the graph is captured on and replayed
  hipStream_t owned_st_ = nullptr;    // created when the caller's stream is the default one
  hipEvent_t order_ev_ = nullptr;
  // k_final's meshes come from a device table (several meshes)
  bool force_final_table_ = false;
  bool final_table(const FinalTable& T) const { return T.segs.size() > 1 || (force_final_table_ && !T.empty()); }
  void add_final_seg(FinalTable& T, int l, int job, const SegDesc& m, const float4* P1, float4* positions);
  void launch_final_table(int l, FinalTable& T, bool ids, const char* stage);
  void launch_deep(int l, FinalTable& T);
  LakTable lak_;
  void plan_blocks(FinalTable& T, bool quad, bool deep);
  void set_final_table(FinalView& V, const FinalTable& T) const;
  // single mesh: the first level's edge numbering ran during the analysis
  // read-back (the level then launches its face points only)
  bool number_early_ = false;
  // ... and, when the first level feeds another, its face points, into the
  // first level's position buffer allocated before the read-back
  bool early_faces_ = false;
  float4* early_p1_ = nullptr;
  int64_t early_p1_cap_ = 0;
  std::vector<int> faceless_;  // jobs without faces
};

std::string flags_message(int f);

}  // namespace slak
