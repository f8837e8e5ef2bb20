// Host engine: device context, resident protein spectra, ligand tables and
// the two search pipelines (reference dataflow and fused/pruned).
#pragma once
#include <hip/hip_runtime.h>

#include <array>
#include <atomic>
#include <cstdint>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "cdk_types.hpp"

namespace cdk {

// Error carrying a C-ABI status code.
struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

enum Status {
  kOk = 0,
  kErrInvalid = 1,
  kErrHip = 2,
  kErrNoMem = 3,
  kErrUnsupported = 4,
  kErrPending = 5,
  kErrBudget = 6,
  kErrCancelled = 7,
};

void hip_check(hipError_t e, const char* what);

// Grow-only device buffer.
struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf();
  void ensure(size_t bytes);
  void release();
  template <class T> T* as() const { return static_cast<T*>(p); }
};

// Part of a device allocation.
struct DevView {
  void* p = nullptr;
  template <class T> T* as() const { return static_cast<T*>(p); }
};

struct Context;

// One call's use of its context's scratch memory (the context lock held for
// the object's life): a device arena and a pinned host arena that grow to what
// a call needs and stay with the context for the next, up to its scratch_keep
// bytes and half as many; a call that needed more gives its arena back when it
// ends.
// A call that ends by an exception waits for the stream first, so nothing
// queued still reads or writes the arenas.
class CallScratch {
 public:
  explicit CallScratch(Context& c);
  ~CallScratch();
  CallScratch(const CallScratch&) = delete;
  CallScratch& operator=(const CallScratch&) = delete;
  // The arena's start, at least `bytes` long; once per call each.
  char* dev(size_t bytes);
  char* host(size_t bytes);
  // Host memory of the caller to device memory and back through pinned
  // slots, the host's copy of one piece beside the transfer of another
  // (a copy straight from or to pageable memory stages the same bytes with no
  // overlap).  in() leaves the last transfers queued on the context stream;
  // out() returns when dst is written.  Both use the host arena.
  void in(void* dev_dst, const void* src, size_t bytes);
  void out(void* dst, const void* dev_src, size_t bytes);

 private:
  Context& ctx_;
  int exceptions_;
};

// Offsets of the 256-byte aligned parts of an arena.
struct Layout {
  size_t end = 0;
  size_t add(size_t bytes) {
    const size_t o = end;
    end += (bytes + 255) & ~(size_t)255;
    return o;
  }
};

// Resident protein: potential grids and their forward spectra, all channels,
// FP32, [channel][X][Y][Z] and [channel][X][Y][Z/2+1] (NoMini:177-199).
struct Protein {
  Context* ctx = nullptr;
  int nch = 0;  // num grids: vdW channels + 1 elec (ReadGrids.cpp:27)
  int N = 0;
  float h = 0.f;
  float mid[3] = {0, 0, 0};
  float len[3] = {0, 0, 0};
  std::vector<float> radii;  // nch - 1 probe radii
  DevBuf mem[5];             // the memory of the arrays below, one block or one each
  DevView grid;              // float [nch][G]
  DevView spec;              // float2 [nch][H]
  DevView spec_lb;           // the same spectra in the fused engine's line-blocked layout
  DevView spec_kz;           // and in the column form's kz-plane layout (grid edge 64 only)
  DevView spec_mf;           // and in the atom form's matrix-core layout (grid edges 64, 96 and 128)
  size_t G() const { return (size_t)N * N * N; }
  size_t H() const { return (size_t)N * N * (N / 2 + 1); }
  // gridMin = mid - len / 2 evaluated in float, then widened (NoMini:149-151).
  double grid_min(int k) const { return (double)(mid[k] - len[k] / 2); }
};

// Ligand with its channel assignment against a protein's probe radii
// (GetIdxOfAtomsForVdwRadius.cpp:4-35).
struct Ligand {
  int natom = 0;
  std::vector<float> charge, eps, radius;
  int num_vdw_used = 0;
  std::vector<int> idx_vdw_used;               // used probe indices, ascending
  std::vector<std::vector<int>> atoms_of_radius;  // per probe radius, ascending atom indices
  std::vector<int> atom_channel;               // per atom: ligand vdW channel index
  // kernel-side tables for this ligand alone (list_off = w_off = 0)
  LigandDesc desc{};
  std::vector<int> chan_atoms;
  std::vector<int> pad_atoms;  // chan_atoms with each channel padded to a multiple of 8 by -1
  std::vector<float> wv, wq;
  int nch() const { return num_vdw_used + 1; }
};

std::unique_ptr<Ligand> make_ligand(const Protein& p, int natom, const float* charge, const float* eps,
                                    const float* radius);

// One docking job: a ligand, its conformers and per-conformer quaternions.
struct Job {
  const Ligand* lig = nullptr;
  int nconf = 0;
  const float* coords = nullptr;  // [nconf][natom][3]
  int nquat = 0;
  const float* quats = nullptr;   // [nconf][nquat][4]
  bool shared_quats = false;      // one quaternion set [nquat][4] for every conformer
  // Pose range [pose_begin, pose_end) in [conformer][quaternion] order.
  size_t pose_begin = 0;
  size_t pose_end = ~(size_t)0;
  size_t npose() const {
    const size_t n = (size_t)nconf * nquat;
    const size_t e = pose_end < n ? pose_end : n;
    return e > pose_begin ? e - pose_begin : 0;
  }
};

// Per-pose result over a job's pose range, [conformer][quaternion] order.
struct PoseResults {
  std::vector<float> energy;   // +inf when the window is empty
  std::vector<int> index;      // [n][3] best translation (i, j, k); -1 when empty
  std::vector<float> mincoor;  // [n][3]
  std::vector<int> box;        // [n][3] occupied ligand box (max grid index + 2)
  std::vector<int> win;        // [n][3] translation window
};

enum Engine { kEngineReference = 0, kEngineFused = 1 };

struct StageTimes {
  double ms[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int launches[8] = {0, 0, 0, 0, 0, 0, 0, 0};
};

// Search tables resident on the device (ligand table, channel lists,
// weights, conformer coordinates, pose slots, results) plus an optional
// hipGraph of the whole fused launch sequence.
struct Prepared {
  const Protein* prot = nullptr;
  std::vector<LigandDesc> ligs;
  std::vector<int> chan, pad;
  std::vector<float> wv, wq, coords;
  std::vector<PoseSlot> slots;
  std::vector<size_t> job_first, job_n;
  int astride = 0, cmax = 0, boxmax = 2, max_chan_atoms = 1;
  int dummy_lig = 0;
  // one device allocation: the tables (uploaded as one piece), then the keys
  // and the per-pose metadata (copied back as one piece, `res_bytes` from
  // d_keys on, the metadata res_meta bytes in)
  DevBuf d_all;
  DevView d_ligs, d_chan, d_pad, d_wv, d_wq, d_coords, d_slots, d_keys, d_meta;
  size_t res_bytes = 0, res_meta = 0;
  bool ran = false;  // executed since it was built
  hipGraphExec_t graph = nullptr;
  uint64_t graph_gen = 0;
  size_t graph_chunk = 0;
  int graph_group = 0, graph_fwd = -1, graph_inv = -1, graph_depth = 0, graph_poses = 0, graph_pipe = -1,
      graph_products = -1, graph_overlap = -1;
  std::vector<PoseResults> results;
  void* h_up = nullptr;  // pinned staging of the tables' upload
  size_t h_up_cap = 0;
  bool h_up_busy = false;  // its last upload may still be queued
  void* h_res = nullptr;   // pinned staging of the results
  size_t h_res_cap = 0;
  // Pipelined callers (the server): `done` marks the end of the launch
  // sequence on the context stream (`start` the first launch), so the host can
  // build the next table while this one runs.
  hipEvent_t start = nullptr, done = nullptr;
  Prepared() = default;
  Prepared(const Prepared&) = delete;
  Prepared& operator=(const Prepared&) = delete;
  ~Prepared();
  void drop_graph();
};

struct Context {
  int device = 0;
  hipStream_t stream = nullptr;
  // The atom form's z-inverse stage of launch set i runs here, overlapped
  // with set i + 1's mid stage on `stream` (two T2 buffers; the ordering
  // events, two per launch set, are created before any capture).
  hipStream_t stream_z = nullptr;
  std::vector<hipEvent_t> set_events;
  std::mutex mu;
  std::map<int, DevBuf*> twiddles;
  // options
  size_t ws_budget = 8ull << 30;  // bytes of per-batch working arrays
  int ref_batch = 50;             // poses per reference-dataflow batch (NoMini:208)
  int fused_chunk = 0;            // 0 = from budget
  int mid_group = 0;              // poses per mid-stage workgroup; 0 = by launch size
  int mid_depth = 0;              // mid-stage register ring depth with a fixed group; 0 = 2
  int mid_poses = 0;              // poses sharing each protein load in the mid stage with a fixed group; 0 = 1
  int pipeline = -1;              // fused pipeline form (kPipePlanes, kPipeColumns, kPipeAtoms); -1 = chosen once per grid edge
  int overlap_z = 1;              // atom form: overlap each launch set's z-inverse stage with the next set
  int atom_products = 2;          // atom form products: kAtomF16x3 (exact 3-part FP16 splits), kAtomF16, kAtomF32
  int fwd_variant = -1;           // forward plane stage form; -1 = by grid edge
  int inv_variant = -1;           // inverse plane stage form; -1 = by grid edge
  bool use_graph = true;
  bool time_stages = false;
  size_t max_dyn_lds = 64 * 1024;
  // The pipeline form taken, per grid edge: the forms round differently, so it
  // is chosen once and kept for the context's life (results then do not depend
  // on how poses are batched).
  std::map<int, int> tuned_pipe;
  int last_fwd = -1, last_inv = -1, last_group = 0, last_depth = 0, last_poses = 0,
      last_pipe = -1;
  StageTimes stage_times;
  // Launch-set working arrays: one pool, never above ws_budget (unless
  // fused_chunk is forced), carved per search into the rotated atoms, atom
  // placements, A (ligand or product spectra), T (correlation spectra, the
  // atom form's T2) and the overlapped atom form's second T2 buffer.
  // ws_generation counts reallocations and re-carvings, so a captured graph
  // that baked in the old addresses is rebuilt.
  DevBuf d_pool;
  float* w_rot = nullptr;
  AtomGrid* w_ag = nullptr;
  float2* w_A = nullptr;
  float2* w_T = nullptr;
  float2* w_T2b = nullptr;
  // the reference dataflow's batch arrays
  DevBuf d_L, d_Lhat, d_S, d_E;
  uint64_t ws_generation = 1;
  // scratch of the synchronous calls (CallScratch)
  DevBuf call_dev;
  void* call_host = nullptr;
  size_t call_host_cap = 0;
  std::vector<hipEvent_t> call_events;
  // Most bytes the device arena keeps between calls; the host arena and each
  // buffer of the idle tables keep half as many.
  std::atomic<size_t> scratch_keep{128ull << 20};
  // Tables of finished cdk_search calls, kept for the next ones: at most
  // kIdleSearches of them.  Every call takes one for itself, so calls of
  // several threads never share one.
  static constexpr size_t kIdleSearches = 2;
  std::mutex idle_mu;
  std::vector<std::unique_ptr<Prepared>> idle;

  explicit Context(int dev);
  ~Context();
  const float2* twiddle(int N);
  // Device and pinned host bytes kept for the synchronous calls, and those
  // above scratch_keep given back (context lock held).
  size_t scratch_bytes();
  void trim_scratch();
  void trim_call_arenas();
  bool may_keep(const Prepared& t) const;
};

void protein_upload(Protein& p, int nch, int N, float h, const float* mid, const float* len, const float* radii,
                    const float* values);
// Builds the potential grids on the device from atoms (gridbuild.hip), then
// the spectra as protein_upload does.
void protein_build(Protein& p, int natom, const double* xyz, const double* charge, const double* epsilon,
                   const double* radius, int nprobe, const float* probe_radii, int N, float h, const float* mid,
                   const float* len, double lj_cutoff, double elec_cutoff, double lj_cap, double elec_cap);

// Largest job (in launch sets) captured as one hipGraph; larger jobs launch
// eagerly.
constexpr size_t kMaxGraphSets = 2048;

// Builds and uploads the tables of a set of jobs (inputs resident in HBM).
void prepare_search(Context& ctx, const Protein& prot, const std::vector<Job>& jobs, Prepared& t);
// Runs every prepared pose; results land in t.results (one entry per job).
// With use_graph the fused launch sequence is captured once and replayed.
void execute_search(Context& ctx, Prepared& t, Engine engine, bool use_graph);
// The same in pipelined pieces: build_search fills t's host tables (no
// device work, no lock); submit_search uploads them and enqueues the fused
// launch sequence and the result copies on the context stream without
// waiting (t's host tables must stay unchanged until finish_search);
// finish_search waits for t's sequence and decodes
// t.results.  Successive submissions run in stream order.
void build_search(const Protein& prot, const std::vector<Job>& jobs, Prepared& t);
void submit_search(Context& ctx, Prepared& t);
void finish_search(Context& ctx, Prepared& t);
// GPU milliseconds of t's last submitted sequence (after finish_search).
float search_gpu_ms(Prepared& t);
// prepare + execute without a graph, one job; results straight to the caller's
// arrays (index and mincoor optional).
void run_search(Context& ctx, const Protein& prot, const Job& job, Engine engine, float* energy, int* index,
                float* mincoor);

// Grid score of explicit poses (FP64 trilinear, see rescore.hip): coords
// [npose][natom][3] in A; energy [npose]; grad [npose][natom][3] and inside
// [npose] optional.  refine_poses moves each pose rigidly downhill in place.
void rescore_poses(Context& ctx, const Protein& prot, const Ligand& lig, int npose, const double* coords,
                   double* energy, double* grad, int* inside);
void refine_poses(Context& ctx, const Protein& prot, const Ligand& lig, int npose, double* coords, int steps,
                  double penalty, double* energy);

// Random-torsion conformers on the device (conformers.hip): every trial sets
// the rotors in order to angles from a (seed, trial, rotor) stream; trials
// passing the steric filter are kept in trial order, at most max_keep.
// Returns the number kept; out [max_keep][natom][3], trial_index [max_keep].
int generate_conformers(Context& ctx, int natom, const double* coords, int nrotor, const int* rotors,
                        const unsigned char* moving, const unsigned char* exclude, int ntrial, uint64_t seed,
                        double clash_dist, int max_keep, double* out, int* trial_index);

// Retained-pose export (export.cpp).
std::string pose_file_name(int conformer, int rank);
std::string energy_row(int conformer, int rank, float energy);
void write_poses(const char* dir, int conformer, int n, int natom, const double* poses, const float* energy,
                 const char* const* names, const char* const* elements, const char* energy_path);
// One protein channel in OpenMM's x-fastest order (double) and the grid
// bounds in nm: min x, y, z then max x, y, z.
void grid_for_openmm(Context& ctx, const Protein& prot, int channel, double* values, double* bounds_nm);

// Decode helpers shared with tests.
float key_energy(unsigned long long key);
unsigned key_index(unsigned long long key);

}  // namespace cdk
