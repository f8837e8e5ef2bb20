// Host engine: device context, resident protein spectra, ligand tables and
// the two search pipelines.
#include "engine.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>

#include "conformers.hpp"
#include "gridbuild.hpp"
#include "kernels.hpp"
#include "noalloc.hpp"
#include "rescore.hpp"

namespace cdk {

void hip_check(hipError_t e, const char* what) {
  if (e == hipSuccess) return;
  const std::string msg = std::string(what) + ": " + hipGetErrorString(e);
  if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation) throw Error(kErrNoMem, msg);
  throw Error(kErrHip, msg);
}

DevBuf::~DevBuf() { release(); }

void DevBuf::release() {
  if (p) (void)hipFree(p);
  p = nullptr;
  cap = 0;
}

void DevBuf::ensure(size_t bytes) {
  if (bytes <= cap) return;
  release();
  if (bytes == 0) return;
  hip_check(hipMalloc(&p, bytes), "hipMalloc");
  cap = bytes;
}

Context::Context(int dev) : device(dev) {
  int n = 0;
  hip_check(hipGetDeviceCount(&n), "hipGetDeviceCount");
  if (dev < 0 || dev >= n) throw Error(kErrInvalid, "device index out of range");
  hip_check(hipSetDevice(dev), "hipSetDevice");
  hip_check(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking), "hipStreamCreate");
  hip_check(hipStreamCreateWithFlags(&stream_z, hipStreamNonBlocking), "hipStreamCreate");
  int lds = 0;
  hip_check(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev), "hipDeviceGetAttribute");
  max_dyn_lds = (size_t)lds;
  hip_check(configure_fwd_reg(max_dyn_lds), "configure forward kernels");
  // the device address of this device's fixed no-alloc array, once per device
  hip_check(noalloc_init(dev), "no-alloc scratch address");
}

Context::~Context() {
  (void)hipSetDevice(device);
  if (stream) (void)hipStreamSynchronize(stream);
  if (stream_z) (void)hipStreamSynchronize(stream_z);
  for (auto& kv : twiddles) delete kv.second;
  idle.clear();
  if (call_host) (void)hipHostFree(call_host);
  for (hipEvent_t e : call_events) (void)hipEventDestroy(e);
  for (hipEvent_t e : set_events) (void)hipEventDestroy(e);
  if (stream_z) (void)hipStreamDestroy(stream_z);
  if (stream) (void)hipStreamDestroy(stream);
}

const float2* Context::twiddle(int N) {
  auto it = twiddles.find(N);
  if (it != twiddles.end()) return it->second->as<float2>();
  std::vector<float2> t(N);
  const double two_pi = 6.283185307179586476925286766559;
  for (int m = 0; m < N; ++m) {
    const double a = two_pi * (double)m / (double)N;
    t[m] = make_float2((float)std::cos(a), (float)-std::sin(a));
  }
  auto* b = new DevBuf();
  b->ensure(N * sizeof(float2));
  hip_check(hipMemcpy(b->p, t.data(), N * sizeof(float2), hipMemcpyHostToDevice), "twiddle upload");
  twiddles[N] = b;
  return b->as<float2>();
}

CallScratch::CallScratch(Context& c) : ctx_(c), exceptions_(std::uncaught_exceptions()) {}

CallScratch::~CallScratch() {
  if (std::uncaught_exceptions() > exceptions_) (void)hipStreamSynchronize(ctx_.stream);
  ctx_.trim_call_arenas();
}

void Context::trim_call_arenas() {
  const size_t keep = scratch_keep;
  const bool dev_over = call_dev.cap > keep, host_over = call_host_cap > keep / 2;
  if (dev_over || host_over) (void)hipStreamSynchronize(stream);
  if (dev_over) call_dev.release();
  if (host_over) {
    (void)hipHostFree(call_host);
    call_host = nullptr;
    call_host_cap = 0;
  }
}

bool Context::may_keep(const Prepared& t) const {
  const size_t most = scratch_keep / 2;
  return t.d_all.cap <= most && t.h_up_cap <= most && t.h_res_cap <= most;
}

void Context::trim_scratch() {
  trim_call_arenas();
  std::lock_guard<std::mutex> lock(idle_mu);
  idle.erase(std::remove_if(idle.begin(), idle.end(), [&](const auto& t) { return !may_keep(*t); }), idle.end());
}

size_t Context::scratch_bytes() {
  size_t n = call_dev.cap + call_host_cap;
  std::lock_guard<std::mutex> lock(idle_mu);
  for (const auto& t : idle) n += t->d_all.cap + t->h_up_cap + t->h_res_cap;
  return n;
}

char* CallScratch::dev(size_t bytes) {
  if (bytes > ctx_.call_dev.cap) {
    hip_check(hipStreamSynchronize(ctx_.stream), "hipStreamSynchronize");
    ctx_.call_dev.ensure((bytes + 0xffff) & ~(size_t)0xffff);
  }
  return ctx_.call_dev.as<char>();
}

char* CallScratch::host(size_t bytes) {
  if (bytes > ctx_.call_host_cap) {
    hip_check(hipStreamSynchronize(ctx_.stream), "hipStreamSynchronize");  // its last transfers
    if (ctx_.call_host) (void)hipHostFree(ctx_.call_host);
    ctx_.call_host = nullptr;
    ctx_.call_host_cap = 0;
    bytes = (bytes + 0xffff) & ~(size_t)0xffff;
    // coherent: kernels read and write it in place
    hip_check(hipHostMalloc(&ctx_.call_host, bytes, hipHostMallocCoherent), "hipHostMalloc");
    ctx_.call_host_cap = bytes;
  }
  return static_cast<char*>(ctx_.call_host);
}

namespace {

// Pieces of the copies.  Measured for 9.4 MB: down 336 us in 1 MB pieces (367
// in 2 MB, 430 in 512 KB, 485 in one, 540 from pageable memory), up 350 us in
// 2 MB pieces with the spectra after it (387 in 1 MB, 408 in one).
constexpr size_t kDownPiece = 1ull << 20, kUpPiece = 2ull << 20;
constexpr size_t kPieceBytes = 16ull << 20;  // of the host arena, all pieces in flight
constexpr size_t kMaxPieces = kPieceBytes / kDownPiece;

void slot_events(Context& c) {
  while (c.call_events.size() < kMaxPieces) {
    hipEvent_t e = nullptr;
    hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
    c.call_events.push_back(e);
  }
}

}  // namespace

void CallScratch::in(void* dev_dst, const void* src, size_t bytes) {
  if (!bytes) return;
  slot_events(ctx_);
  constexpr size_t kSlotBytes = kUpPiece, kSlots = kPieceBytes / kUpPiece;
  const size_t n = (bytes + kSlotBytes - 1) / kSlotBytes;
  char* h = host(std::min(n, kSlots) * kSlotBytes);
  for (size_t i = 0; i < n; ++i) {
    char* slot = h + (i % kSlots) * kSlotBytes;
    const size_t o = i * kSlotBytes, len = std::min(kSlotBytes, bytes - o);
    if (i >= kSlots) hip_check(hipEventSynchronize(ctx_.call_events[i % kSlots]), "upload slot");
    std::memcpy(slot, static_cast<const char*>(src) + o, len);
    hip_check(hipMemcpyAsync(static_cast<char*>(dev_dst) + o, slot, len, hipMemcpyHostToDevice, ctx_.stream), "H2D");
    if (n > kSlots) hip_check(hipEventRecord(ctx_.call_events[i % kSlots], ctx_.stream), "hipEventRecord");
  }
}

void CallScratch::out(void* dst, const void* dev_src, size_t bytes) {
  if (!bytes) return;
  if (bytes <= kDownPiece) {  // one piece: 139 KB 16 us, with an event for the wait 22; 460 KB 28, 35
    char* p = host(kDownPiece);
    hip_check(hipMemcpyAsync(p, dev_src, bytes, hipMemcpyDeviceToHost, ctx_.stream), "D2H");
    hip_check(hipStreamSynchronize(ctx_.stream), "D2H sync");
    std::memcpy(dst, p, bytes);
    return;
  }
  slot_events(ctx_);
  constexpr size_t kSlotBytes = kDownPiece, kSlots = kPieceBytes / kDownPiece;
  const size_t n = (bytes + kSlotBytes - 1) / kSlotBytes;
  char* h = host(std::min(n, kSlots) * kSlotBytes);
  auto fetch = [&](size_t i) {
    const size_t o = i * kSlotBytes, len = std::min(kSlotBytes, bytes - o);
    hip_check(hipMemcpyAsync(h + (i % kSlots) * kSlotBytes, static_cast<const char*>(dev_src) + o, len,
                             hipMemcpyDeviceToHost, ctx_.stream),
              "D2H");
    hip_check(hipEventRecord(ctx_.call_events[i % kSlots], ctx_.stream), "hipEventRecord");
  };
  for (size_t i = 0; i < std::min(n, kSlots); ++i) fetch(i);
  for (size_t i = 0; i < n; ++i) {
    const size_t o = i * kSlotBytes, len = std::min(kSlotBytes, bytes - o);
    hip_check(hipEventSynchronize(ctx_.call_events[i % kSlots]), "download slot");
    std::memcpy(static_cast<char*>(dst) + o, h + (i % kSlots) * kSlotBytes, len);
    if (i + kSlots < n) fetch(i + kSlots);
  }
}

namespace {

void protein_setup(Protein& p, int nch, int N, float h, const float* mid, const float* len, const float* radii) {
  if (nch < 2 || nch > kMaxCh) throw Error(kErrInvalid, "number of grids must be in [2, 16]");
  if (!grid_edge_supported(N)) throw Error(kErrUnsupported, "grid edge must be one of 32, 48, 64, 96, 128");
  if (!(h > 0.f)) throw Error(kErrInvalid, "grid spacing must be positive");
  p.nch = nch;
  p.N = N;
  p.h = h;
  for (int k = 0; k < 3; ++k) {
    p.mid[k] = mid ? mid[k] : 0.f;
    p.len[k] = len ? len[k] : (float)(N - 1) * h;
  }
  p.radii.assign(radii, radii + (nch - 1));
  // One allocation, unless every array is below 2 MB (32^3 up to 15 channels):
  // those are made and freed out of memory the runtime holds.  Measured, upload
  // and close, one allocation / one per array: 32 (9 channels) 118 / 77 us, 48
  // 203 / 225, 64 337 / 414.
  const size_t H = (size_t)nch * p.H() * sizeof(float2);
  const size_t bytes[5] = {(size_t)nch * p.G() * sizeof(float), H, H, col_supported(N) ? H : 0,
                           atoms_supported(N) ? H : 0};
  DevView* const views[5] = {&p.grid, &p.spec, &p.spec_lb, &p.spec_kz, &p.spec_mf};
  if (*std::max_element(bytes, bytes + 5) < (2u << 20)) {
    for (int i = 0; i < 5; ++i) {
      p.mem[i].ensure(bytes[i]);
      views[i]->p = p.mem[i].p;
    }
    return;
  }
  Layout l;
  size_t off[5];
  for (int i = 0; i < 5; ++i) off[i] = l.add(bytes[i]);
  p.mem[0].ensure(l.end);
  for (int i = 0; i < 5; ++i) views[i]->p = bytes[i] ? p.mem[0].as<char>() + off[i] : nullptr;
}

// Forward R2C of every channel (NoMini:177-199) plus the copies the fused
// mid stages read (line-blocked; kz-plane blocks at grid edge 64, matrix-core
// blocks at 64, 96 and 128).
void protein_spectra(Protein& p) {
  Context& ctx = *p.ctx;
  hip_check(launch_r2c_3d(ctx.stream, p.N, p.grid.as<float>(), p.spec.as<float2>(), p.nch, ctx.twiddle(p.N)),
            "protein R2C");
  hip_check(launch_to_line_blocks(ctx.stream, p.N, p.spec.as<float2>(), p.spec_lb.as<float2>(), p.nch),
            "protein spectra line blocks");
  if (col_supported(p.N)) {
    hip_check(launch_to_kz_blocks(ctx.stream, p.N, p.spec.as<float2>(), p.spec_kz.as<float2>(), p.nch),
              "protein spectra kz blocks");
  }
  if (atoms_supported(p.N)) {
    hip_check(launch_to_mfma_blocks(ctx.stream, p.N, p.spec.as<float2>(), p.spec_mf.as<float2>(), p.nch),
              "protein spectra matrix-core blocks");
  }
  hip_check(hipStreamSynchronize(ctx.stream), "protein R2C sync");
}

}  // namespace

void protein_upload(Protein& p, int nch, int N, float h, const float* mid, const float* len, const float* radii,
                    const float* values) {
  protein_setup(p, nch, N, h, mid, len, radii);
  Context& ctx = *p.ctx;
  CallScratch scratch(ctx);
  scratch.in(p.grid.p, values, (size_t)nch * p.G() * sizeof(float));
  protein_spectra(p);
}

void protein_build(Protein& p, int natom, const double* xyz, const double* charge, const double* epsilon,
                   const double* radius, int nprobe, const float* probe_radii, int N, float h, const float* mid,
                   const float* len, double lj_cutoff, double elec_cutoff, double lj_cap, double elec_cap) {
  if (natom < 0 || nprobe < 1 || nprobe > grid_build_max_probes())
    throw Error(kErrInvalid, "atom count must be >= 0 and probe count in [1, 15]");
  protein_setup(p, nprobe + 1, N, h, mid, len, probe_radii);
  Context& ctx = *p.ctx;
  CallScratch scratch(ctx);
  Layout l;
  const size_t o_atoms = l.add((size_t)std::max(natom, 1) * 6 * sizeof(double));
  const size_t o_probe = l.add((size_t)nprobe * sizeof(double));
  char* hs = scratch.host(l.end);
  char* ds = scratch.dev(l.end);
  double* atoms = reinterpret_cast<double*>(hs + o_atoms);
  for (int i = 0; i < natom; ++i) {
    for (int k = 0; k < 3; ++k) atoms[(size_t)i * 6 + k] = xyz[i * 3 + k];
    atoms[(size_t)i * 6 + 3] = charge[i];
    atoms[(size_t)i * 6 + 4] = radius[i];
    atoms[(size_t)i * 6 + 5] = epsilon[i];
  }
  std::copy(probe_radii, probe_radii + nprobe, reinterpret_cast<double*>(hs + o_probe));
  hip_check(hipMemcpyAsync(ds, hs, l.end, hipMemcpyHostToDevice, ctx.stream), "atoms H2D");
  const double gmin[3] = {p.grid_min(0), p.grid_min(1), p.grid_min(2)};
  hip_check(launch_build_grids(ctx.stream, natom, reinterpret_cast<const double*>(ds + o_atoms), nprobe,
                               reinterpret_cast<const double*>(ds + o_probe), N, gmin,
                               (double)h, lj_cutoff, elec_cutoff, lj_cap, elec_cap, p.grid.as<float>()),
            "build grids");
  protein_spectra(p);
}

std::unique_ptr<Ligand> make_ligand(const Protein& p, int natom, const float* charge, const float* eps,
                                    const float* radius) {
  if (natom <= 0 || natom > kMaxAtoms) throw Error(kErrInvalid, "ligand atom count must be in [1, 512]");
  auto L = std::make_unique<Ligand>();
  L->natom = natom;
  L->charge.assign(charge, charge + natom);
  L->eps.assign(eps, eps + natom);
  L->radius.assign(radius, radius + natom);
  const int nv = p.nch - 1;
  // GetIdxOfAtomsForVdwRadius.cpp:9-23: nearest probe radius, strict '<' so
  // the first of equal distances wins; float difference, double running min.
  L->atoms_of_radius.assign(nv, {});
  L->atom_channel.assign(natom, 0);
  std::vector<int> radius_of_atom(natom);
  for (int i = 0; i < natom; ++i) {
    int idx = 0;
    double diff = std::abs(radius[i] - p.radii[0]);
    for (int j = 1; j < nv; ++j) {
      if (std::abs(radius[i] - p.radii[j]) < diff) {
        idx = j;
        diff = std::abs(radius[i] - p.radii[j]);
      }
    }
    L->atoms_of_radius[idx].push_back(i);
    radius_of_atom[i] = idx;
  }
  // GetIdxOfAtomsForVdwRadius.cpp:26-34: used radii in ascending order.
  for (int j = 0; j < nv; ++j)
    if (!L->atoms_of_radius[j].empty()) L->idx_vdw_used.push_back(j);
  L->num_vdw_used = (int)L->idx_vdw_used.size();
  const int nch = L->num_vdw_used + 1;
  if (nch > kMaxCh) throw Error(kErrInvalid, "too many channels");
  LigandDesc& d = L->desc;
  std::memset(&d, 0, sizeof(d));
  d.natom = natom;
  d.nch = nch;
  d.w_off = 0;
  d.list_off = 0;
  int pos = 0;
  for (int c = 0; c < L->num_vdw_used; ++c) {
    d.ch_start[c] = pos;
    d.pmap[c] = L->idx_vdw_used[c];
    for (int a : L->atoms_of_radius[L->idx_vdw_used[c]]) {
      L->chan_atoms.push_back(a);
      L->atom_channel[a] = c;
    }
    pos = (int)L->chan_atoms.size();
  }
  // Electrostatic channel: every atom, elec protein grid is the last one
  // (TranRotaConfSearchNoMini.cu:143-146).
  d.ch_start[L->num_vdw_used] = pos;
  d.pmap[L->num_vdw_used] = p.nch - 1;
  for (int a = 0; a < natom; ++a) L->chan_atoms.push_back(a);
  d.ch_start[nch] = (int)L->chan_atoms.size();
  d.pad_off = 0;
  for (int c = 0; c < nch; ++c) {
    d.pad_start[c] = (int)L->pad_atoms.size();
    L->pad_atoms.insert(L->pad_atoms.end(), L->chan_atoms.begin() + d.ch_start[c],
                        L->chan_atoms.begin() + d.ch_start[c + 1]);
    while (L->pad_atoms.size() % 8) L->pad_atoms.push_back(-1);
  }
  d.pad_start[nch] = (int)L->pad_atoms.size();
  L->wv.resize(natom);
  L->wq.resize(natom);
  float wmax = 0.f;
  for (int a = 0; a < natom; ++a) {
    L->wv[a] = std::sqrt(eps[a]);  // float overload, as FillLigandGrid.cpp:45
    L->wq[a] = charge[a];
    if (!std::isfinite(L->wv[a]) || !std::isfinite(L->wq[a])) throw Error(kErrInvalid, "non-finite atom weight");
    wmax = std::max({wmax, std::abs(L->wv[a]), std::abs(L->wq[a])});
  }
  // wmax * 2^e in [2^12, 2^13): e = 13 - exponent of wmax (frexp: wmax = m 2^x, m in [0.5, 1))
  int ex = 0;
  if (wmax > 0.f) (void)std::frexp(wmax, &ex);
  const int e = wmax > 0.f ? std::max(-100, std::min(100, 13 - ex)) : 0;
  d.ascale = std::ldexp(1.f, e);
  d.aunscale = std::ldexp(1.f, -e);
  return L;
}

float key_energy(unsigned long long key) {
  if (key == ~0ull) return std::numeric_limits<float>::infinity();
  unsigned u = (unsigned)(key >> 32);
  u = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}

unsigned key_index(unsigned long long key) { return (unsigned)(key & 0xffffffffu); }

namespace {

// Upper bound of the occupied box edge of a conformer over all rotations:
// the extent along any axis is at most the largest pairwise distance.
int box_bound(const float* xyz, int natom, float h, int N, double qscale) {
  double d2 = 0;
  for (int i = 0; i < natom; ++i)
    for (int j = i + 1; j < natom; ++j) {
      double s = 0;
      for (int k = 0; k < 3; ++k) {
        const double d = (double)xyz[i * 3 + k] - (double)xyz[j * 3 + k];
        s += d * d;
      }
      d2 = std::max(d2, s);
    }
  const int b = (int)std::floor(std::sqrt(d2) * qscale / (double)h) + 3;
  return std::min(N, std::max(b, 2));
}

// Rotation scales lengths by |q|^2; the bound must hold for non-unit input.
double quat_scale(const float* q, size_t n) {
  double m = 1.0;
  for (size_t i = 0; i < n; ++i) {
    const double s = (double)q[i * 4] * q[i * 4] + (double)q[i * 4 + 1] * q[i * 4 + 1] +
                     (double)q[i * 4 + 2] * q[i * 4 + 2] + (double)q[i * 4 + 3] * q[i * 4 + 3];
    m = std::max(m, s);
  }
  return m * (1.0 + 1e-5);
}

void build_tables(const Protein& prot, const std::vector<Job>& jobs, Prepared& t) {
  std::map<const Ligand*, int> lig_index;
  for (const Job& j : jobs) {
    if (!j.lig) throw Error(kErrInvalid, "job without ligand");
    if (j.nconf < 0 || j.nquat < 0) throw Error(kErrInvalid, "negative conformer or quaternion count");
    if (lig_index.count(j.lig)) continue;
    const Ligand& L = *j.lig;
    LigandDesc d = L.desc;
    d.list_off = (int)t.chan.size();
    d.pad_off = (int)t.pad.size();
    d.w_off = (int)t.wv.size();
    t.chan.insert(t.chan.end(), L.chan_atoms.begin(), L.chan_atoms.end());
    t.pad.insert(t.pad.end(), L.pad_atoms.begin(), L.pad_atoms.end());
    t.wv.insert(t.wv.end(), L.wv.begin(), L.wv.end());
    t.wq.insert(t.wq.end(), L.wq.begin(), L.wq.end());
    for (int c = 0; c < d.nch; ++c)
      if (d.pmap[c] < 0 || d.pmap[c] >= prot.nch) throw Error(kErrInvalid, "ligand built for another protein");
    lig_index[j.lig] = (int)t.ligs.size();
    t.ligs.push_back(d);
    t.astride = std::max(t.astride, L.natom);
    t.cmax = std::max(t.cmax, d.nch);
    for (int c = 0; c < d.nch; ++c) t.max_chan_atoms = std::max(t.max_chan_atoms, d.ch_start[c + 1] - d.ch_start[c]);
  }
  // Padding ligand: zero atoms, so its poses are never valid.
  LigandDesc dummy;
  std::memset(&dummy, 0, sizeof(dummy));
  dummy.nch = 1;
  dummy.ascale = dummy.aunscale = 1.f;
  t.dummy_lig = (int)t.ligs.size();
  t.ligs.push_back(dummy);
  if (t.chan.empty()) t.chan.push_back(0);
  if (t.wv.empty()) {
    t.wv.push_back(0.f);
    t.wq.push_back(0.f);
  }
  size_t nslots = 0;
  for (const Job& j : jobs) nslots += j.npose();
  if (nslots > (size_t)std::numeric_limits<int>::max()) throw Error(kErrInvalid, "too many poses in one call");
  t.slots.reserve(nslots);
  for (const Job& j : jobs) {
    t.job_first.push_back(t.slots.size());
    const size_t np = j.npose();
    if (np == 0) continue;
    const int li = lig_index[j.lig];
    const int na = j.lig->natom;
    const size_t nq_total = (size_t)(j.shared_quats ? 1 : j.nconf) * j.nquat;
    for (size_t i = 0; i < nq_total * 4; ++i)
      if (!std::isfinite(j.quats[i])) throw Error(kErrInvalid, "non-finite quaternion");
    const double qscale = quat_scale(j.quats, nq_total);
    int cur_conf = -1;
    int off = 0;
    for (size_t pose = j.pose_begin; pose < j.pose_begin + np; ++pose) {
      const int c = (int)(pose / (size_t)j.nquat), r = (int)(pose % (size_t)j.nquat);
      if (c != cur_conf) {
        cur_conf = c;
        if (t.coords.size() + (size_t)na * 3 > (size_t)std::numeric_limits<int>::max())
          throw Error(kErrInvalid, "coordinate table too large");
        off = (int)t.coords.size();
        const float* xyz = j.coords + (size_t)c * na * 3;
        for (int a = 0; a < na * 3; ++a)
          if (!std::isfinite(xyz[a])) throw Error(kErrInvalid, "non-finite ligand coordinate");
        t.coords.insert(t.coords.end(), xyz, xyz + (size_t)na * 3);
        t.boxmax = std::max(t.boxmax, box_bound(xyz, na, prot.h, prot.N, qscale));
      }
      const float* q = j.shared_quats ? j.quats : j.quats + (size_t)c * j.nquat * 4;
      PoseSlot sl;
      std::memset(&sl, 0, sizeof(sl));
      for (int k = 0; k < 4; ++k) sl.q[k] = q[r * 4 + k];
      sl.lig = li;
      sl.coord_off = off;
      t.slots.push_back(sl);
    }
  }
  if (t.coords.empty()) t.coords.resize(3, 0.f);
  t.astride = std::max(t.astride, 1);
  t.cmax = std::max(t.cmax, 1);
}


struct EventTimer {
  Context& ctx;
  std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> ev;
  explicit EventTimer(Context& c) : ctx(c) {}
  ~EventTimer() {
    for (auto& e : ev) {
      (void)hipEventDestroy(e.second.first);
      (void)hipEventDestroy(e.second.second);
    }
  }
  hipEvent_t begin(int stage) {
    if (!ctx.time_stages) return nullptr;
    hipEvent_t a, b;
    hip_check(hipEventCreate(&a), "hipEventCreate");
    hip_check(hipEventCreate(&b), "hipEventCreate");
    ev.push_back({stage, {a, b}});
    hip_check(hipEventRecord(a, ctx.stream), "hipEventRecord");
    return b;
  }
  void end(hipEvent_t b) {
    if (b) hip_check(hipEventRecord(b, ctx.stream), "hipEventRecord");
  }
  void collect() {
    for (auto& e : ev) {
      float ms = 0.f;
      hip_check(hipEventElapsedTime(&ms, e.second.first, e.second.second), "hipEventElapsedTime");
      ctx.stage_times.ms[e.first] += ms;
      ctx.stage_times.launches[e.first] += 1;
    }
  }
};

}  // namespace

namespace {

// Before a working array is reallocated: the context's queued work (a
// server's earlier launch set may still run on either stream) is done with
// the old memory.
void drain_streams(Context& ctx) {
  hip_check(hipStreamSynchronize(ctx.stream), "hipStreamSynchronize");
  hip_check(hipStreamSynchronize(ctx.stream_z), "hipStreamSynchronize");
}

void ensure_work(Context& ctx, size_t bytes_needed, DevBuf& b) {
  if (b.cap >= bytes_needed) return;
  drain_streams(ctx);
  b.ensure(bytes_needed);
  ++ctx.ws_generation;
}

// Carves the five launch-set arrays for `chunk` poses (bytes per pose
// per[i]: rotated atoms, placements, A, T, second T2) from the pool, each
// 256-byte aligned, growing the pool if needed.
void carve_work(Context& ctx, size_t chunk, const size_t (&per)[5]) {
  size_t off[5], end = 0;
  for (int i = 0; i < 5; ++i) {
    off[i] = end;
    end += (chunk * per[i] + 255) & ~(size_t)255;
  }
  if (ctx.d_pool.cap < end) {
    drain_streams(ctx);
    ctx.d_pool.ensure(end);
    ++ctx.ws_generation;
  }
  char* base = static_cast<char*>(ctx.d_pool.p);
  float* rot = reinterpret_cast<float*>(base + off[0]);
  AtomGrid* ag = reinterpret_cast<AtomGrid*>(base + off[1]);
  float2* A = reinterpret_cast<float2*>(base + off[2]);
  float2* T = reinterpret_cast<float2*>(base + off[3]);
  float2* T2b = per[4] ? reinterpret_cast<float2*>(base + off[4]) : nullptr;
  if (rot != ctx.w_rot || ag != ctx.w_ag || A != ctx.w_A || T != ctx.w_T || T2b != ctx.w_T2b) ++ctx.ws_generation;
  ctx.w_rot = rot;
  ctx.w_ag = ag;
  ctx.w_A = A;
  ctx.w_T = T;
  ctx.w_T2b = T2b;
}

// Reference dataflow: one launch sequence per batch of <= B rotations of one
// conformer (TranRotaConfSearchNoMini.cu:385-464).
void enqueue_reference(Context& ctx, const Protein& prot, Prepared& t, EventTimer& timer) {
  const int N = prot.N;
  const size_t G = prot.G(), H = prot.H();
  const float2* tw = ctx.twiddle(N);
  const int B = std::max(1, ctx.ref_batch);
  const int C = t.cmax;
  const size_t per[5] = {(size_t)t.astride * 3 * sizeof(float), (size_t)t.astride * sizeof(AtomGrid), 0, 0, 0};
  carve_work(ctx, (size_t)B, per);
  ensure_work(ctx, (size_t)B * C * G * sizeof(float), ctx.d_L);
  ensure_work(ctx, (size_t)B * C * H * sizeof(float2), ctx.d_Lhat);
  ensure_work(ctx, (size_t)B * H * sizeof(float2), ctx.d_S);
  ensure_work(ctx, (size_t)B * G * sizeof(float), ctx.d_E);
  const PoseSlot* d_slots = t.d_slots.as<PoseSlot>();
  const LigandDesc* d_ligs = t.d_ligs.as<LigandDesc>();
  unsigned long long* d_keys = t.d_keys.as<unsigned long long>();
  RotMeta* d_meta = t.d_meta.as<RotMeta>();
  const size_t total = t.slots.size();
  size_t s = 0;
  while (s < total) {
    const int lig_idx = t.slots[s].lig;
    const int coff = t.slots[s].coord_off;
    size_t e2 = s + 1;
    while (e2 < total && (int)(e2 - s) < B && t.slots[e2].coord_off == coff && t.slots[e2].lig == lig_idx) ++e2;
    const int n = (int)(e2 - s);
    const int nch = t.ligs[lig_idx].nch;
    const int* pmap = reinterpret_cast<const int*>(reinterpret_cast<const char*>(d_ligs + lig_idx) +
                                                   offsetof(LigandDesc, pmap));
    const PoseSlot* sl = d_slots + s;
    hipEvent_t e;
    e = timer.begin(0);
    hip_check(launch_prep(ctx.stream, sl, n, d_ligs, t.d_coords.as<float>(), N, prot.h, t.astride, N,
                          ctx.w_rot, ctx.w_ag, d_meta + s, d_keys + s),
              "prep");
    timer.end(e);
    e = timer.begin(1);
    hip_check(launch_spread_full(ctx.stream, sl, n, d_ligs, t.d_chan.as<int>(), t.d_wv.as<float>(), t.d_wq.as<float>(),
                                 ctx.w_ag, t.astride, d_meta + s, N, nch, ctx.d_L.as<float>()),
              "spread");
    timer.end(e);
    e = timer.begin(2);
    hip_check(launch_r2c_3d(ctx.stream, N, ctx.d_L.as<float>(), ctx.d_Lhat.as<float2>(), n * nch, tw), "ligand R2C");
    timer.end(e);
    e = timer.begin(3);
    hip_check(launch_conj_mult(ctx.stream, ctx.d_Lhat.as<float2>(), prot.spec.as<float2>(), pmap, nch, (long long)H,
                               n),
              "ConjMult");
    timer.end(e);
    e = timer.begin(4);
    hip_check(launch_sum_grids(ctx.stream, ctx.d_Lhat.as<float2>(), ctx.d_S.as<float2>(), nch, (long long)H, n,
                               (float)G),
              "SumGrids");
    timer.end(e);
    e = timer.begin(5);
    hip_check(launch_c2r_3d(ctx.stream, N, ctx.d_S.as<float2>(), ctx.d_E.as<float>(), n, tw), "C2R");
    timer.end(e);
    e = timer.begin(6);
    hip_check(launch_argmin_full(ctx.stream, ctx.d_E.as<float>(), d_meta + s, d_keys + s, N, n), "argmin");
    timer.end(e);
    s = e2;
  }
}

// Whether a fused search on this protein may run the atom form with its
// z-inverse stage overlapped (two T2 buffers).
bool overlap_possible(const Context& ctx, const Protein& prot) {
  return ctx.overlap_z && !ctx.time_stages && atoms_supported(prot.N) && prot.spec_mf.p != nullptr &&
         (ctx.pipeline < 0 || ctx.pipeline == kPipeAtoms);
}

// Bytes per pose of each launch-set working array: rotated atoms, atom
// placements, A (the plane and column forms' ligand spectra), T (correlation
// spectra, the atom form's T2: at grid edges 96 and 128 the window's y rows
// of the product spectra), and the overlapped atom form's second T2 buffer
// when that form may run.
void per_pose_bytes(const Context& ctx, const Protein& prot, const Prepared& t, size_t (&s)[5]) {
  const int N = prot.N, ZH = N / 2 + 1;
  const size_t plane = (size_t)N * ZH;
  s[0] = (size_t)t.astride * 3 * sizeof(float);
  s[1] = (size_t)t.astride * sizeof(AtomGrid);
  s[2] = (size_t)t.cmax * t.boxmax * plane * sizeof(float2);
  s[3] = (size_t)N * plane * sizeof(float2);
  s[4] = overlap_possible(ctx, prot) ? s[3] : 0;
}

// Poses per launch set: as many as the working arrays of the search allow
// within ws_budget (or the forced fused_chunk), at most the search's poses.
size_t fused_chunk(Context& ctx, const Protein& prot, const Prepared& t) {
  if (ctx.fused_chunk > 0) return std::min((size_t)ctx.fused_chunk, std::max<size_t>(t.slots.size(), 1));
  size_t s[5];
  per_pose_bytes(ctx, prot, t, s);
  size_t per = 0;
  for (int i = 0; i < 5; ++i) per += s[i];
  // each array's start is 256-byte aligned: 5 x 256 bytes of slack
  const size_t room = ctx.ws_budget > 5 * 256 ? ctx.ws_budget - 5 * 256 : 0;
  const size_t chunk = std::max<size_t>(1, room / std::max<size_t>(per, 1));
  return std::min(chunk, std::max<size_t>(t.slots.size(), 1));
}

// The launch-set working arrays for `chunk` poses carved from the pool
// (grown when a search needs more; the pool is never larger than the largest
// search's need, so at most ws_budget).
void ensure_fused_work(Context& ctx, const Protein& prot, const Prepared& t, size_t chunk) {
  size_t s[5];
  per_pose_bytes(ctx, prot, t, s);
  carve_work(ctx, chunk, s);
}

struct Tuned {
  int pipe = kPipePlanes;
  int fwd = kFwdBlock, inv = kInvBlock, group = 1, depth = 1, poses = 1;  // plane form
  int col_group = 1;                                                      // column form
  int atom_group = 1;                                                     // atom form
  int mid_group() const { return pipe == kPipeColumns ? col_group : pipe == kPipeAtoms ? atom_group : group; }
};

// Searches whose largest ligand has at most this many atoms take the atom form
// where it is supported, untimed (with FP16 products): it is the fastest for
// them at every edge and launch size.  Measured, us of a call, atom / best other form: 64 24 atoms, 1
// pose 74 / 80, 1,000 1,040 / 1,573; 84 atoms, 20 105 / 252, 400 531 / 1,075;
// 96 40 atoms, 1 93 / 179, 1,000 5,150 / 9,979; 84 atoms, 400 2,769 / 7,090;
// 128 50 atoms, 1 94 / 202, 1,000 10.9 / 29.6 ms; at worst 64 with one atom, 200
// poses 10% behind the column form.  Above it the line depends on the ligand's
// extent: 64, 400 poses, 100 atoms in a chain 837 / 1,431, in a ball of 11 A
// 881 / 743; 200 in a ball 1,410 / 835; 96 4,941 / 4,130.
constexpr int kAtomFormAtoms = 84;

// The forms and the first launch set's schedule of a search.
//  - The pipeline form, once per grid size: the forms round differently, so
//    one per (context, N) keeps results independent of how poses are batched.
//    Searches of larger ligands than kAtomFormAtoms time the forms on their
//    first launch set, twice each, and keep the fastest.
//  - The plane form's forward and inverse stages, which round differently too,
//    by the grid edge.  Measured, us of block / register transforms: 32 (16
//    atoms) forward 20 poses 24 / 23, 4,000 326 / 397, inverse 10 / 21 and 311 /
//    767; 48 (60 atoms) 151 / 157, 3,536 / 5,008 and 10 / 24, 244 / 820; 64 (24
//    atoms) 77 / 51, 4,000 2,586 / 2,668 and 24 / 20, 2,232 / 1,457; 96 (40)
//    1,000 2,755 / 2,140 and 3,571 / 2,689; 128 (50) 10.0 / 6.2 ms and 13.4 /
//    7.3 ms.
//  - The mid stage's schedule by launch size (mid_plan, atom_group); the column
//    form runs one pose per workgroup (24 atoms, us of 1 / 2 / 4 / 8: 10 poses
//    31 / 44 / 84 / 161, 200 207 / 213 / 236 / 274, 8,000 1,578 / 1,584 / 1,571
//    / 1,606 per launch set).  Schedules only reorder work; results are
//    bit-identical.
Tuned tune_fused(Context& ctx, const Protein& prot, Prepared& t, size_t chunk) {
  const int N = prot.N;
  Tuned tu;
  const bool col_ok = col_supported(N) && prot.spec_kz.p != nullptr;
  const bool atoms_ok = atoms_supported(N) && prot.spec_mf.p != nullptr;
  const int n = (int)std::min(chunk, t.slots.size());  // poses of a full launch set
  tu.fwd = (ctx.fwd_variant >= 0 ? ctx.fwd_variant == kFwdReg : N >= 64) && fwd_reg_supported(N) ? kFwdReg : kFwdBlock;
  tu.inv = (ctx.inv_variant >= 0 ? ctx.inv_variant == kInvReg : N >= 64) && inv_reg_supported(N) ? kInvReg : kInvBlock;
  if (ctx.mid_group > 0) {
    const int max_depth = mid_max_depth(N);
    tu.group = ctx.mid_group;
    tu.depth = ctx.mid_depth > 0 ? std::min(ctx.mid_depth, max_depth) : std::min(2, max_depth);
    tu.poses = ctx.mid_poses > 0 ? std::min(ctx.mid_poses, mid_max_poses(N)) : 1;
    tu.col_group = ctx.mid_group;
    tu.atom_group = ctx.mid_group;
  } else {
    const MidPlan mp = mid_plan(N, n);
    tu.group = mp.group;
    tu.depth = mp.depth;
    tu.poses = mp.poses;
    tu.atom_group = atom_group(N, ctx.atom_products, t.astride, n);
  }
  if (ctx.pipeline >= 0) {
    tu.pipe = (ctx.pipeline == kPipeColumns && col_ok)  ? kPipeColumns
              : (ctx.pipeline == kPipeAtoms && atoms_ok) ? kPipeAtoms
                                                         : kPipePlanes;
    return tu;
  }
  auto it = ctx.tuned_pipe.find(N);
  if (it != ctx.tuned_pipe.end()) {
    tu.pipe = it->second;
    return tu;
  }
  if (!col_ok && !atoms_ok) {
    ctx.tuned_pipe[N] = tu.pipe = kPipePlanes;
    return tu;
  }
  if (atoms_ok && ctx.atom_products != kAtomF32 && t.astride <= kAtomFormAtoms) {
    ctx.tuned_pipe[N] = tu.pipe = kPipeAtoms;
    return tu;
  }

  const float2* tw = ctx.twiddle(N);
  const PoseSlot* sl = t.d_slots.as<PoseSlot>();
  const LigandDesc* d_ligs = t.d_ligs.as<LigandDesc>();
  RotMeta* d_meta = t.d_meta.as<RotMeta>();
  unsigned long long* d_keys = t.d_keys.as<unsigned long long>();
  const float invG = 1.0f / (float)prot.G();
  hip_check(launch_prep(ctx.stream, sl, n, d_ligs, t.d_coords.as<float>(), N, prot.h, t.astride, t.boxmax,
                        ctx.w_rot, ctx.w_ag, d_meta, d_keys),
            "tune prep");
  hipEvent_t e0, e1;
  hip_check(hipEventCreate(&e0), "hipEventCreate");
  hip_check(hipEventCreate(&e1), "hipEventCreate");
  auto timed = [&](auto&& launch) {
    float best = 1e30f;
    for (int rep = 0; rep < 2; ++rep) {
      hip_check(hipEventRecord(e0, ctx.stream), "hipEventRecord");
      launch();
      hip_check(hipEventRecord(e1, ctx.stream), "hipEventRecord");
      hip_check(hipEventSynchronize(e1), "hipEventSynchronize");
      float ms = 0.f;
      hip_check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
      best = std::min(best, ms);
    }
    return best;
  };
  try {
    tu.pipe = kPipePlanes;
    float best = timed([&] {
      hip_check(launch_fwd_planes(ctx.stream, N, tu.fwd, sl, n, d_ligs, t.d_chan.as<int>(), t.d_wv.as<float>(),
                                  t.d_wq.as<float>(), ctx.w_ag, t.astride, d_meta, t.cmax, t.boxmax,
                                  t.max_chan_atoms, ctx.w_A, tw),
                "tune fwd planes");
    });
    best += timed([&] {
      hip_check(launch_mid(ctx.stream, N, tu.depth, tu.poses, sl, d_ligs, d_meta, n, tu.group, ctx.w_A, t.cmax,
                           t.boxmax, prot.spec_lb.as<float2>(), prot.nch, ctx.w_T, invG, tw),
                "tune mid");
    });
    best += timed([&] {
      hip_check(launch_inv_argmin(ctx.stream, N, tu.inv, d_meta, n, N - 2, ctx.w_T, d_keys, tw), "tune inverse");
    });
    if (col_ok) {
      float ms = timed([&] {
        hip_check(launch_fwd_z(ctx.stream, N, sl, n, d_ligs, t.d_chan.as<int>(), t.d_wv.as<float>(),
                               t.d_wq.as<float>(), ctx.w_ag, t.astride, d_meta, t.cmax, t.boxmax,
                               t.max_chan_atoms, ctx.w_A, tw),
                  "tune column forward");
      });
      ms += timed([&] {
        hip_check(launch_mid_kz(ctx.stream, N, sl, d_ligs, d_meta, n, tu.col_group, ctx.w_A, t.cmax, t.boxmax,
                                prot.spec_kz.as<float2>(), ctx.w_T, invG, tw),
                  "tune column mid");
      });
      ms += timed([&] {
        hip_check(launch_inv_z(ctx.stream, N, d_meta, n, ctx.w_T, d_keys, tw), "tune column inverse");
      });
      if (ms < best) {
        best = ms;
        tu.pipe = kPipeColumns;
      }
    }
    if (atoms_ok) {
      float ms = timed([&] {
        hip_check(launch_mid_atoms(ctx.stream, N, sl, d_ligs, t.d_pad.as<int>(), t.d_wv.as<float>(),
                                   t.d_wq.as<float>(), ctx.w_ag, t.astride, d_meta, n, tu.atom_group,
                                   prot.spec_mf.as<float2>(), ctx.w_T, invG, tw, ctx.atom_products),
                  "tune atom mid");
      });
      ms += timed([&] {
        hip_check(launch_inv_z(ctx.stream, N, d_meta, n, ctx.w_T, d_keys, tw), "tune atom inverse");
      });
      if (ms < best) tu.pipe = kPipeAtoms;
    }
    ctx.tuned_pipe[N] = tu.pipe;
  } catch (...) {
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    throw;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return tu;
}

// The atom form's z-inverse stage runs on its own stream, one launch set
// behind (not when stages are timed: their events are on the launch stream).
bool overlap_z_stage(const Context& ctx, const Tuned& tu) {
  return tu.pipe == kPipeAtoms && ctx.overlap_z && !ctx.time_stages;
}

// The ordering events of an overlapped search (its second T2 buffer is
// carved with the other arrays), made before any capture.
void ensure_overlap(Context& ctx, const Prepared& t, size_t chunk) {
  if (!ctx.w_T2b) throw Error(kErrInvalid, "overlapped z-inverse stage without its second buffer");
  const size_t sets = (t.slots.size() + chunk - 1) / chunk;
  while (ctx.set_events.size() < 2 * sets) {
    hipEvent_t e = nullptr;
    hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
    ctx.set_events.push_back(e);
  }
}

// Fused pipeline: four launches per chunk of poses, any mix of ligands, in
// the plane or the column form.
void enqueue_fused(Context& ctx, const Protein& prot, Prepared& t, size_t chunk, const Tuned& tu,
                   EventTimer& timer) {
  const int N = prot.N;
  const size_t G = prot.G();
  const float2* tw = ctx.twiddle(N);
  const PoseSlot* d_slots = t.d_slots.as<PoseSlot>();
  const LigandDesc* d_ligs = t.d_ligs.as<LigandDesc>();
  unsigned long long* d_keys = t.d_keys.as<unsigned long long>();
  RotMeta* d_meta = t.d_meta.as<RotMeta>();
  const size_t total = t.slots.size();
  const bool ovl = overlap_z_stage(ctx, tu);
  size_t last_set = 0;
  for (size_t s = 0; s < total; s += chunk) {
    const int n = (int)std::min(chunk, total - s);
    const PoseSlot* sl = d_slots + s;
    const size_t si = s / chunk;  // launch set index
    hipEvent_t e;
    e = timer.begin(0);
    hip_check(launch_prep(ctx.stream, sl, n, d_ligs, t.d_coords.as<float>(), N, prot.h, t.astride, t.boxmax,
                          ctx.w_rot, ctx.w_ag, d_meta + s, d_keys + s),
              "prep");
    timer.end(e);
    if (tu.pipe == kPipeAtoms) {
      // overlapped: T2 alternates between two buffers; set si's mid stage
      // waits for set si - 2's z-inverse, the last reader of its buffer
      float2* T2 = ovl && (si & 1) ? ctx.w_T2b : ctx.w_T;
      if (ovl && si >= 2) hip_check(hipStreamWaitEvent(ctx.stream, ctx.set_events[2 * (si - 2) + 1], 0), "wait");
      e = timer.begin(2);
      hip_check(launch_mid_atoms(ctx.stream, N, sl, d_ligs, t.d_pad.as<int>(), t.d_wv.as<float>(),
                                 t.d_wq.as<float>(), ctx.w_ag, t.astride, d_meta + s, n,
                                 ctx.mid_group > 0 ? ctx.mid_group : atom_group(N, ctx.atom_products, t.astride, n),
                                 prot.spec_mf.as<float2>(), T2, 1.0f / (float)G, tw, ctx.atom_products),
                "atom mid");
      timer.end(e);
      if (ovl) {
        hip_check(hipEventRecord(ctx.set_events[2 * si], ctx.stream), "record");
        hip_check(hipStreamWaitEvent(ctx.stream_z, ctx.set_events[2 * si], 0), "wait");
        hip_check(launch_inv_z(ctx.stream_z, N, d_meta + s, n, T2, d_keys + s, tw), "atom inverse + argmin");
        hip_check(hipEventRecord(ctx.set_events[2 * si + 1], ctx.stream_z), "record");
        last_set = si;
      } else {
        e = timer.begin(3);
        hip_check(launch_inv_z(ctx.stream, N, d_meta + s, n, T2, d_keys + s, tw), "atom inverse + argmin");
        timer.end(e);
      }
      continue;
    }
    if (tu.pipe == kPipeColumns) {
      e = timer.begin(1);
      hip_check(launch_fwd_z(ctx.stream, N, sl, n, d_ligs, t.d_chan.as<int>(), t.d_wv.as<float>(),
                             t.d_wq.as<float>(), ctx.w_ag, t.astride, d_meta + s, t.cmax, t.boxmax,
                             t.max_chan_atoms, ctx.w_A, tw),
                "column forward");
      timer.end(e);
      e = timer.begin(2);
      hip_check(launch_mid_kz(ctx.stream, N, sl, d_ligs, d_meta + s, n, tu.col_group, ctx.w_A, t.cmax,
                              t.boxmax, prot.spec_kz.as<float2>(), ctx.w_T, 1.0f / (float)G, tw),
                "column mid");
      timer.end(e);
      e = timer.begin(3);
      hip_check(launch_inv_z(ctx.stream, N, d_meta + s, n, ctx.w_T, d_keys + s, tw),
                "column inverse + argmin");
      timer.end(e);
      continue;
    }
    e = timer.begin(1);
    hip_check(launch_fwd_planes(ctx.stream, N, tu.fwd, sl, n, d_ligs, t.d_chan.as<int>(), t.d_wv.as<float>(),
                                t.d_wq.as<float>(), ctx.w_ag, t.astride, d_meta + s, t.cmax, t.boxmax,
                                t.max_chan_atoms, ctx.w_A, tw),
              "fwd planes");
    timer.end(e);
    e = timer.begin(2);
    const MidPlan mp = ctx.mid_group > 0 ? MidPlan{tu.group, tu.depth, tu.poses} : mid_plan(N, n);
    hip_check(launch_mid(ctx.stream, N, mp.depth, mp.poses, sl, d_ligs, d_meta + s, n, mp.group, ctx.w_A, t.cmax,
                         t.boxmax,
                         prot.spec_lb.as<float2>(), prot.nch, ctx.w_T, 1.0f / (float)G, tw),
              "mid");
    timer.end(e);
    e = timer.begin(3);
    hip_check(launch_inv_argmin(ctx.stream, N, tu.inv, d_meta + s, n, N - 2, ctx.w_T, d_keys + s, tw),
              "inverse + argmin");
    timer.end(e);
  }
  // join: the last two sets' z-inverse stages (earlier ones are ordered
  // before later mid stages) back into the launch stream
  if (ovl) {
    for (size_t si = last_set > 0 ? last_set - 1 : 0; si <= last_set; ++si)
      hip_check(hipStreamWaitEvent(ctx.stream, ctx.set_events[2 * si + 1], 0), "join");
  }
}

}  // namespace

Prepared::~Prepared() {
  drop_graph();
  if (h_up) (void)hipHostFree(h_up);
  if (h_res) (void)hipHostFree(h_res);
  if (start) (void)hipEventDestroy(start);
  if (done) (void)hipEventDestroy(done);
}

void Prepared::drop_graph() {
  if (graph) (void)hipGraphExecDestroy(graph);
  graph = nullptr;
}

void build_search(const Protein& prot, const std::vector<Job>& jobs, Prepared& t) {
  t.drop_graph();
  t.ligs.clear();
  t.chan.clear();
  t.pad.clear();
  t.wv.clear();
  t.wq.clear();
  t.coords.clear();
  t.slots.clear();
  t.job_first.clear();
  t.job_n.clear();
  t.astride = 0;
  t.cmax = 0;
  t.boxmax = 2;
  t.max_chan_atoms = 1;
  build_tables(prot, jobs, t);
  for (const Job& j : jobs) t.job_n.push_back(j.npose());
  t.prot = &prot;
  t.ran = false;
}

namespace {

// t's tables to the device on the context stream (context lock held): through
// t's pinned staging in one asynchronous copy (one from pageable memory would
// hold the host until the stream's earlier work is done), the staging rewritten
// only once that copy is over; or through `scratch` in pieces.
void upload_tables(Context& ctx, Prepared& t, CallScratch* scratch = nullptr) {
  struct Part {
    DevView* dst;
    const void* src;
    size_t bytes, off;
  };
  Part parts[7] = {{&t.d_ligs, t.ligs.data(), t.ligs.size() * sizeof(LigandDesc), 0},
                   {&t.d_chan, t.chan.data(), t.chan.size() * sizeof(int), 0},
                   {&t.d_pad, t.pad.data(), t.pad.size() * sizeof(int), 0},
                   {&t.d_wv, t.wv.data(), t.wv.size() * sizeof(float), 0},
                   {&t.d_wq, t.wq.data(), t.wq.size() * sizeof(float), 0},
                   {&t.d_coords, t.coords.data(), t.coords.size() * sizeof(float), 0},
                   {&t.d_slots, t.slots.data(), t.slots.size() * sizeof(PoseSlot), 0}};
  Layout l;
  for (Part& p : parts) p.off = l.add(std::max<size_t>(p.bytes, 4));
  const size_t tables = l.end, total = std::max<size_t>(t.slots.size(), 1);
  const size_t keys = l.add(total * sizeof(unsigned long long));
  const size_t meta = l.add(total * sizeof(RotMeta));
  if (t.h_up_busy) hip_check(hipStreamSynchronize(ctx.stream), "upload sync");
  t.h_up_busy = false;
  if (!scratch && tables > t.h_up_cap) {
    if (t.h_up) (void)hipHostFree(t.h_up);
    t.h_up = nullptr;
    t.h_up_cap = 0;
    hip_check(hipHostMalloc(&t.h_up, tables), "hipHostMalloc");
    t.h_up_cap = tables;
  }
  t.d_all.ensure(l.end);
  char* d = t.d_all.as<char>();
  char* h = static_cast<char*>(t.h_up);
  for (const Part& p : parts) {
    p.dst->p = d + p.off;
    if (!p.bytes) continue;
    if (scratch) {
      scratch->in(p.dst->p, p.src, p.bytes);
      hip_check(hipStreamSynchronize(ctx.stream), "tables H2D");  // the next part reuses the pieces
    } else {
      std::memcpy(h + p.off, p.src, p.bytes);
    }
  }
  if (!scratch) {
    hip_check(hipMemcpyAsync(d, h, tables, hipMemcpyHostToDevice, ctx.stream), "tables H2D");
    t.h_up_busy = true;
  }
  t.d_keys.p = d + keys;
  t.d_meta.p = d + meta;
  t.res_meta = meta - keys;
  t.res_bytes = t.res_meta + total * sizeof(RotMeta);
}

}  // namespace

void prepare_search(Context& ctx, const Protein& prot, const std::vector<Job>& jobs, Prepared& t) {
  build_search(prot, jobs, t);
  std::lock_guard<std::mutex> lock(ctx.mu);
  hip_check(hipSetDevice(ctx.device), "hipSetDevice");
  upload_tables(ctx, t);
}

namespace {

// Enqueues t's launch sequence (context lock held).
void enqueue_search(Context& ctx, Prepared& t, Engine engine, bool use_graph, EventTimer& timer,
                    hipEvent_t start = nullptr) {
  const Protein& prot = *t.prot;
  const size_t total = t.slots.size();
  if (engine == kEngineReference) {
    if (start) hip_check(hipEventRecord(start, ctx.stream), "hipEventRecord");
    enqueue_reference(ctx, prot, t, timer);
  } else {
    const size_t chunk = fused_chunk(ctx, prot, t);
    ensure_fused_work(ctx, prot, t, chunk);
    (void)ctx.twiddle(prot.N);
    const Tuned tu = tune_fused(ctx, prot, t, chunk);
    ctx.last_fwd = tu.fwd;
    ctx.last_inv = tu.inv;
    ctx.last_pipe = tu.pipe;
    ctx.last_group = tu.mid_group();
    ctx.last_depth = tu.depth;
    ctx.last_poses = tu.poses;
    const int ovl = overlap_z_stage(ctx, tu) ? 1 : 0;
    if (ovl) ensure_overlap(ctx, t, chunk);
    if (start) hip_check(hipEventRecord(start, ctx.stream), "hipEventRecord");
    // Jobs of more launch sets than kMaxGraphSets run eagerly: a host
    // segmentation fault inside the search of a 3.28 M-pose uneven batch
    // captured as one graph of 3 410 launch sets (3 304 had passed) has no
    // cause found in this code, so graphs stay at sizes that have run.
    const size_t nsets = (total + chunk - 1) / chunk;
    if (use_graph && !ctx.time_stages && nsets <= kMaxGraphSets) {
      if (!t.graph || t.graph_gen != ctx.ws_generation || t.graph_chunk != chunk || t.graph_group != tu.mid_group() ||
          t.graph_fwd != tu.fwd || t.graph_inv != tu.inv || t.graph_depth != tu.depth ||
          t.graph_poses != tu.poses || t.graph_pipe != tu.pipe || t.graph_products != ctx.atom_products ||
          t.graph_overlap != ovl) {
        t.drop_graph();
        hipGraph_t g = nullptr;
        hip_check(hipStreamBeginCapture(ctx.stream, hipStreamCaptureModeRelaxed), "hipStreamBeginCapture");
        try {
          enqueue_fused(ctx, prot, t, chunk, tu, timer);
        } catch (...) {
          (void)hipStreamEndCapture(ctx.stream, &g);
          if (g) (void)hipGraphDestroy(g);
          throw;
        }
        hip_check(hipStreamEndCapture(ctx.stream, &g), "hipStreamEndCapture");
        hipError_t ie = hipGraphInstantiate(&t.graph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        hip_check(ie, "hipGraphInstantiate");
        t.graph_gen = ctx.ws_generation;
        t.graph_chunk = chunk;
        t.graph_group = tu.mid_group();
        t.graph_pipe = tu.pipe;
        t.graph_products = ctx.atom_products;
        t.graph_overlap = ovl;
        t.graph_fwd = tu.fwd;
        t.graph_inv = tu.inv;
        t.graph_depth = tu.depth;
        t.graph_poses = tu.poses;
      }
      hip_check(hipGraphLaunch(t.graph, ctx.stream), "hipGraphLaunch");
    } else {
      enqueue_fused(ctx, prot, t, chunk, tu, timer);
    }
  }
}

// Enqueues the copy of t's keys and per-pose metadata to its pinned staging.
void enqueue_results(Context& ctx, Prepared& t) {
  if (t.res_bytes > t.h_res_cap) {
    if (t.h_res) (void)hipHostFree(t.h_res);
    t.h_res = nullptr;
    t.h_res_cap = 0;
    hip_check(hipHostMalloc(&t.h_res, t.res_bytes), "hipHostMalloc");
    t.h_res_cap = t.res_bytes;
  }
  hip_check(hipMemcpyAsync(t.h_res, t.d_keys.p, t.res_bytes, hipMemcpyDeviceToHost, ctx.stream), "results D2H");
}

// n poses' results from their keys and metadata; index, mincoor, box and win
// optional ([n][3] each).
void decode_poses(unsigned N, const unsigned long long* keys, const RotMeta* meta, size_t n, float* energy, int* index,
                  float* mincoor, int* box, int* win) {
  for (size_t i = 0; i < n; ++i) {
    const unsigned long long k = keys[i];
    const RotMeta& m = meta[i];
    const bool found = k != ~0ull && m.valid;
    energy[i] = found ? key_energy(k) : std::numeric_limits<float>::infinity();
    if (index) {
      const unsigned lin = key_index(k);
      index[i * 3 + 0] = found ? (int)(lin / (N * N)) : -1;
      index[i * 3 + 1] = found ? (int)((lin / N) % N) : -1;
      index[i * 3 + 2] = found ? (int)(lin % N) : -1;
    }
    for (int c = 0; c < 3; ++c) {
      if (mincoor) mincoor[i * 3 + c] = m.minc[c];
      if (box) box[i * 3 + c] = m.box[c];
      if (win) win[i * 3 + c] = m.win[c];
    }
  }
}

// t's keys and metadata in its host staging.
const unsigned long long* staged_keys(const Prepared& t) { return static_cast<const unsigned long long*>(t.h_res); }
const RotMeta* staged_meta(const Prepared& t) {
  return reinterpret_cast<const RotMeta*>(static_cast<const char*>(t.h_res) + t.res_meta);
}

void decode_results(Prepared& t) {
  t.results.assign(t.job_first.size(), PoseResults());
  for (size_t j = 0; j < t.job_first.size(); ++j) {
    const size_t n = t.job_n[j];
    PoseResults& r = t.results[j];
    r.energy.resize(n);
    r.index.resize(n * 3);
    r.mincoor.resize(n * 3);
    r.box.resize(n * 3);
    r.win.resize(n * 3);
    const size_t first = t.job_first[j];
    decode_poses((unsigned)t.prot->N, staged_keys(t) + first, staged_meta(t) + first, n, r.energy.data(),
                 r.index.data(), r.mincoor.data(), r.box.data(), r.win.data());
  }
}

// Runs t's launch sequence to its end (context lock held).
void run_prepared(Context& ctx, Prepared& t, Engine engine, bool use_graph) {
  EventTimer timer(ctx);
  enqueue_search(ctx, t, engine, use_graph, timer);
  enqueue_results(ctx, t);
  hip_check(hipStreamSynchronize(ctx.stream), "search sync");
  t.h_up_busy = false;
  t.ran = true;
  timer.collect();
}

// The same with tables too large to keep for the next call: no pinned memory
// of t's own, its results come through the context's arena in pieces, decoded
// beside the next piece's copy.
void run_unstaged(Context& ctx, Prepared& t, Engine engine, CallScratch& scratch, float* energy, int* index,
                  float* mincoor) {
  EventTimer timer(ctx);
  enqueue_search(ctx, t, engine, false, timer);
  constexpr size_t kPer = kDownPiece / (sizeof(unsigned long long) + sizeof(RotMeta)) & ~(size_t)31, kSlots = 4;
  constexpr size_t kSlotBytes = kPer * (sizeof(unsigned long long) + sizeof(RotMeta));
  slot_events(ctx);
  const size_t total = t.slots.size(), n = (total + kPer - 1) / kPer;
  char* h = scratch.host(std::min(n, kSlots) * kSlotBytes);
  auto keys = [&](size_t i) { return reinterpret_cast<unsigned long long*>(h + (i % kSlots) * kSlotBytes); };
  auto meta = [&](size_t i) { return reinterpret_cast<RotMeta*>(keys(i) + kPer); };
  auto fetch = [&](size_t i) {
    const size_t o = i * kPer, len = std::min(kPer, total - o);
    hip_check(hipMemcpyAsync(keys(i), t.d_keys.as<unsigned long long>() + o, len * sizeof(unsigned long long),
                             hipMemcpyDeviceToHost, ctx.stream),
              "keys D2H");
    hip_check(hipMemcpyAsync(meta(i), t.d_meta.as<RotMeta>() + o, len * sizeof(RotMeta), hipMemcpyDeviceToHost,
                             ctx.stream),
              "meta D2H");
    hip_check(hipEventRecord(ctx.call_events[i % kSlots], ctx.stream), "hipEventRecord");
  };
  for (size_t i = 0; i < std::min(n, kSlots); ++i) fetch(i);
  for (size_t i = 0; i < n; ++i) {
    const size_t o = i * kPer, len = std::min(kPer, total - o);
    hip_check(hipEventSynchronize(ctx.call_events[i % kSlots]), "result piece");
    decode_poses((unsigned)t.prot->N, keys(i), meta(i), len, energy + o, index ? index + o * 3 : nullptr,
                 mincoor ? mincoor + o * 3 : nullptr, nullptr, nullptr);
    if (i + kSlots < n) fetch(i + kSlots);
  }
  timer.collect();
}

}  // namespace

void execute_search(Context& ctx, Prepared& t, Engine engine, bool use_graph) {
  std::lock_guard<std::mutex> lock(ctx.mu);
  hip_check(hipSetDevice(ctx.device), "hipSetDevice");
  if (!t.prot) throw Error(kErrInvalid, "search not prepared");
  t.results.assign(t.job_first.size(), PoseResults());
  if (t.slots.empty()) return;
  run_prepared(ctx, t, engine, use_graph);
  decode_results(t);
}

void submit_search(Context& ctx, Prepared& t) {
  std::lock_guard<std::mutex> lock(ctx.mu);
  hip_check(hipSetDevice(ctx.device), "hipSetDevice");
  if (!t.prot) throw Error(kErrInvalid, "search not built");
  if (!t.start) hip_check(hipEventCreate(&t.start), "hipEventCreate");
  if (!t.done) hip_check(hipEventCreate(&t.done), "hipEventCreate");
  upload_tables(ctx, t);
  if (t.slots.empty()) {
    hip_check(hipEventRecord(t.start, ctx.stream), "hipEventRecord");
  } else {
    EventTimer timer(ctx);  // stages are timed only by the synchronous path
    const bool ts = ctx.time_stages;
    ctx.time_stages = false;
    try {
      enqueue_search(ctx, t, kEngineFused, false, timer, t.start);
      enqueue_results(ctx, t);
    } catch (...) {
      ctx.time_stages = ts;
      throw;
    }
    ctx.time_stages = ts;
  }
  hip_check(hipEventRecord(t.done, ctx.stream), "hipEventRecord");
}

void finish_search(Context& ctx, Prepared& t) {
  (void)ctx;
  if (!t.done) throw Error(kErrInvalid, "search not submitted");
  hip_check(hipEventSynchronize(t.done), "search wait");
  t.results.assign(t.job_first.size(), PoseResults());
  t.h_up_busy = false;
  if (!t.slots.empty()) decode_results(t);
}

float search_gpu_ms(Prepared& t) {
  float ms = 0.f;
  if (t.start && t.done) hip_check(hipEventElapsedTime(&ms, t.start, t.done), "hipEventElapsedTime");
  return ms;
}

void run_search(Context& ctx, const Protein& prot, const Job& job, Engine engine, float* energy, int* index,
                float* mincoor) {
  std::unique_ptr<Prepared> t;
  {
    std::lock_guard<std::mutex> lock(ctx.idle_mu);
    if (!ctx.idle.empty()) {
      t = std::move(ctx.idle.back());
      ctx.idle.pop_back();
    }
  }
  if (!t) t = std::make_unique<Prepared>();
  {
    // a call that fails leaves nothing queued that reads t's staging
    struct Drain {
      Context& ctx;
      Prepared& t;
      ~Drain() {
        if (t.h_up_busy) (void)hipStreamSynchronize(ctx.stream);
        t.h_up_busy = false;
      }
    } drain{ctx, *t};
    build_search(prot, {job}, *t);
    std::lock_guard<std::mutex> lock(ctx.mu);
    hip_check(hipSetDevice(ctx.device), "hipSetDevice");
    const size_t n = t->slots.size(), most = ctx.scratch_keep / 2;
    if (n * (sizeof(unsigned long long) + sizeof(RotMeta)) > most) {
      // not kept for the next call: pinned memory of its own would be made and
      // freed by each such call (1 000 000 poses at 32^3 260 -> 247 ms)
      CallScratch scratch(ctx);
      upload_tables(ctx, *t, &scratch);
      run_unstaged(ctx, *t, engine, scratch, energy, index, mincoor);
    } else {
      upload_tables(ctx, *t);
      if (n) {
        run_prepared(ctx, *t, engine, false);
        decode_poses((unsigned)prot.N, staged_keys(*t), staged_meta(*t), n, energy, index, mincoor, nullptr, nullptr);
      }
    }
  }
  t->prot = nullptr;
  std::lock_guard<std::mutex> lock(ctx.idle_mu);
  if (ctx.may_keep(*t) && ctx.idle.size() < Context::kIdleSearches) ctx.idle.push_back(std::move(t));
}

namespace {

// Per-atom protein channel (vdW probe of the atom, -1 if none) and weights.
void atom_channels(const Protein& prot, const Ligand& lig, std::vector<int>& pch) {
  pch.assign(lig.natom, -1);
  for (int a = 0; a < lig.natom; ++a) {
    const int c = lig.atom_channel[a];
    if (c >= 0 && c < lig.num_vdw_used) pch[a] = lig.idx_vdw_used[c];
  }
  (void)prot;
}

// Poses go through the pinned arena in pieces, two slots in turn, so the host
// copies one piece in and another out while the kernel works on a third; the
// kernels read and write the slots in place over the host link.  A call within
// one piece has one slot.  Measured, one slot of 32 MB -> two of 4 MB, 40 atoms:
// 200 000 poses rescored 10.0 -> 7.1 ms, with the gradient 25.7 -> 20.8, 40 000
// refined for 50 steps 8.5 -> 7.5.  Two of 1 / 2 / 8 MB: 7.9 / 7.4 / 7.0 ms, 18.3
// / 17.2 / 20.9, 8.6 / 7.6 / 7.2; small ones leave large poses' kernels short
// (500 poses of 300 atoms refined 0.97 / 0.67 / 0.64 ms, 4 MB 0.61).
struct PoseStage {
  int per = 0;    // poses per piece
  int slots = 1;
  // the ligand's channels and weights, then per slot the poses' coordinates
  // and results
  int* pch = nullptr;
  float *wv = nullptr, *wq = nullptr;
  int* inside[2] = {};
  double *x[2] = {}, *g[2] = {}, *e[2] = {};
};
constexpr size_t kPosePieceBytes = 4ull << 20;

PoseStage stage_poses(CallScratch& scratch, const Protein& prot, const Ligand& lig, int npose, bool grad) {
  const size_t na = (size_t)lig.natom, pose = na * 3 * sizeof(double);
  PoseStage s;
  s.per = (int)std::max<size_t>(1, std::min<size_t>((size_t)npose, kPosePieceBytes / ((grad ? 2 : 1) * pose + 16)));
  s.slots = s.per < npose ? 2 : 1;
  Layout l;
  const size_t o_pch = l.add(na * sizeof(int)), o_wv = l.add(na * sizeof(float)), o_wq = l.add(na * sizeof(float));
  size_t o_e[2], o_in[2], o_x[2], o_g[2];
  for (int i = 0; i < s.slots; ++i) {
    o_e[i] = l.add(s.per * sizeof(double));
    o_in[i] = l.add(s.per * sizeof(int));
    o_x[i] = l.add(s.per * pose);
    o_g[i] = grad ? l.add(s.per * pose) : 0;
  }
  char* h = scratch.host(l.end);
  s.pch = reinterpret_cast<int*>(h + o_pch);
  s.wv = reinterpret_cast<float*>(h + o_wv);
  s.wq = reinterpret_cast<float*>(h + o_wq);
  for (int i = 0; i < s.slots; ++i) {
    s.e[i] = reinterpret_cast<double*>(h + o_e[i]);
    s.inside[i] = reinterpret_cast<int*>(h + o_in[i]);
    s.x[i] = reinterpret_cast<double*>(h + o_x[i]);
    if (grad) s.g[i] = reinterpret_cast<double*>(h + o_g[i]);
  }
  std::vector<int> pch;
  atom_channels(prot, lig, pch);
  for (int a = 0; a < lig.natom; ++a) {
    s.pch[a] = pch[a];
    s.wv[a] = std::sqrt(lig.eps[a]);
    s.wq[a] = lig.charge[a];
  }
  return s;
}

// run(slot, n) for the pieces of npose poses, coords copied in before and
// done(slot, first, n) called after each.
template <class Run, class Done>
void for_pieces(Context& ctx, const PoseStage& w, int npose, size_t per_pose, const double* coords, Run&& run,
                Done&& done) {
  slot_events(ctx);
  int before = 0, first = 0;  // the piece before: its poses and their first
  for (int p0 = 0, i = 0; p0 < npose; ++i) {
    const int n = std::min(w.per, npose - p0), slot = i & 1;
    std::memcpy(w.x[slot], coords + p0 * per_pose, n * per_pose * sizeof(double));
    run(slot, n);
    if (p0 + n < npose) hip_check(hipEventRecord(ctx.call_events[slot], ctx.stream), "hipEventRecord");
    if (i > 0) {
      hip_check(hipEventSynchronize(ctx.call_events[slot ^ 1]), "pose piece");
      done(slot ^ 1, first, before);
    }
    first = p0;
    before = n;
    p0 += n;
    if (p0 == npose) {
      hip_check(hipStreamSynchronize(ctx.stream), "pose pieces");
      done(slot, first, before);
    }
  }
}

}  // namespace

void rescore_poses(Context& ctx, const Protein& prot, const Ligand& lig, int npose, const double* coords,
                   double* energy, double* grad, int* inside) {
  std::lock_guard<std::mutex> lock(ctx.mu);
  hip_check(hipSetDevice(ctx.device), "hipSetDevice");
  if (npose <= 0) return;
  CallScratch scratch(ctx);
  const PoseStage w = stage_poses(scratch, prot, lig, npose, grad != nullptr);
  const double gmin[3] = {prot.grid_min(0), prot.grid_min(1), prot.grid_min(2)};
  const size_t per = (size_t)lig.natom * 3;
  for_pieces(
      ctx, w, npose, per, coords,
      [&](int slot, int n) {
        hip_check(launch_rescore(ctx.stream, n, lig.natom, w.x[slot], w.pch, w.wv, w.wq, prot.grid.as<float>(), prot.N,
                                 prot.nch - 1, gmin, (double)prot.h, w.e[slot], w.g[slot], w.inside[slot]),
                  "rescore");
      },
      [&](int slot, int p0, int n) {
        std::memcpy(energy + p0, w.e[slot], n * sizeof(double));
        if (grad) std::memcpy(grad + p0 * per, w.g[slot], n * per * sizeof(double));
        if (inside) std::memcpy(inside + p0, w.inside[slot], n * sizeof(int));
      });
}

void refine_poses(Context& ctx, const Protein& prot, const Ligand& lig, int npose, double* coords, int steps,
                  double penalty, double* energy) {
  std::lock_guard<std::mutex> lock(ctx.mu);
  hip_check(hipSetDevice(ctx.device), "hipSetDevice");
  if (npose <= 0) return;
  CallScratch scratch(ctx);
  const PoseStage w = stage_poses(scratch, prot, lig, npose, false);
  const double gmin[3] = {prot.grid_min(0), prot.grid_min(1), prot.grid_min(2)};
  const size_t per = (size_t)lig.natom * 3;
  for_pieces(
      ctx, w, npose, per, coords,
      [&](int slot, int n) {
        hip_check(launch_refine(ctx.stream, n, lig.natom, w.x[slot], w.pch, w.wv, w.wq, prot.grid.as<float>(), prot.N,
                                prot.nch - 1, gmin, (double)prot.h, steps, penalty, w.e[slot]),
                  "refine");
      },
      [&](int slot, int p0, int n) {
        std::memcpy(coords + p0 * per, w.x[slot], n * per * sizeof(double));
        std::memcpy(energy + p0, w.e[slot], n * sizeof(double));
      });
}

// Device bytes of a set of conformer trials (512 atoms: 4 096 trials, 101 MB).
constexpr size_t kConformerBytes = 64ull << 20;

int generate_conformers(Context& ctx, int natom, const double* coords, int nrotor, const int* rotors,
                        const unsigned char* moving, const unsigned char* exclude, int ntrial, uint64_t seed,
                        double clash_dist, int max_keep, double* out, int* trial_index) {
  std::lock_guard<std::mutex> lock(ctx.mu);
  hip_check(hipSetDevice(ctx.device), "hipSetDevice");
  if (ntrial <= 0 || max_keep <= 0) return 0;
  for (int r = 0; r < nrotor; ++r)
    for (int k = 0; k < 4; ++k)
      if (rotors[r * 4 + k] < 0 || rotors[r * 4 + k] >= natom) throw Error(kErrInvalid, "rotor atom out of range");
  const size_t per = (size_t)natom * 3;
  const int rw = (nrotor + 63) / 64, ew = (natom + 63) / 64;
  // Trials run a set at a time and stop once enough have passed: the kept
  // ones are the first max_keep in trial order, so later trials cannot
  // matter.  A first set of 4 096 (four wavefronts per SIMD) takes hardly
  // longer than one of a few; the next sets follow the share that passed.  No
  // set is larger than kConformerBytes allow for its trials' coordinates and
  // the kept ones' copies, so a call that keeps most of many trials needs no
  // more memory than another.
  int kept = 0, done = 0;
  const size_t most = std::max<size_t>(4096, kConformerBytes / (2 * std::max<size_t>(per, 1) * sizeof(double)));
  const size_t cap = std::min({(size_t)ntrial, most, (size_t)1 << 16});
  const size_t keep = std::min<size_t>(max_keep, cap);
  int set = (int)std::min(cap, std::max<size_t>(4096, max_keep));
  CallScratch scratch(ctx);
  Layout in, l;
  const size_t o_x = in.add(per * sizeof(double)), o_rot = in.add((size_t)nrotor * 4 * sizeof(int));
  const size_t o_mv = in.add((size_t)rw * natom * 8), o_ex = in.add((size_t)natom * ew * 8);
  l.add(in.end);
  const size_t o_ok = l.add(cap * sizeof(int)), o_list = l.add(keep * sizeof(int));
  const size_t o_count = l.add(sizeof(int)), o_trial = l.add(keep * sizeof(int));
  const size_t o_kept = l.add(keep * per * sizeof(double)), o_all = l.add(cap * per * sizeof(double));
  char* d = scratch.dev(l.end);
  char* h = scratch.host(in.end);
  std::memcpy(h + o_x, coords, per * sizeof(double));
  if (nrotor) std::memcpy(h + o_rot, rotors, (size_t)nrotor * 4 * sizeof(int));
  unsigned long long* mv = reinterpret_cast<unsigned long long*>(h + o_mv);
  unsigned long long* ex = reinterpret_cast<unsigned long long*>(h + o_ex);
  std::fill(mv, mv + (size_t)rw * natom, 0ull);
  std::fill(ex, ex + (size_t)natom * ew, 0ull);
  for (int r = 0; r < nrotor; ++r)
    for (int a = 0; a < natom; ++a)
      if (moving[(size_t)r * natom + a]) mv[(size_t)(r / 64) * natom + a] |= 1ull << (r % 64);
  for (int a = 0; a < natom; ++a)
    for (int b = 0; b < natom; ++b)
      if (exclude[(size_t)a * natom + b]) ex[(size_t)a * ew + b / 64] |= 1ull << (b % 64);
  hip_check(hipMemcpyAsync(d, h, in.end, hipMemcpyHostToDevice, ctx.stream), "conformer inputs H2D");
  while (done < ntrial && kept < max_keep) {
    const int need = std::min(max_keep - kept, set);
    hip_check(launch_conformers(ctx.stream, natom, reinterpret_cast<double*>(d + o_x), nrotor,
                                reinterpret_cast<int*>(d + o_rot), reinterpret_cast<unsigned long long*>(d + o_mv),
                                reinterpret_cast<unsigned long long*>(d + o_ex), done, set, seed, clash_dist,
                                reinterpret_cast<double*>(d + o_all), reinterpret_cast<int*>(d + o_ok)),
              "conformers");
    hip_check(launch_keep_conformers(ctx.stream, natom, done, set, reinterpret_cast<int*>(d + o_ok),
                                     reinterpret_cast<double*>(d + o_all), need, reinterpret_cast<int*>(d + o_list),
                                     reinterpret_cast<int*>(d + o_count), reinterpret_cast<double*>(d + o_kept),
                                     reinterpret_cast<int*>(d + o_trial)),
              "conformers kept");
    int n = 0;
    scratch.out(&n, d + o_count, sizeof(int));
    scratch.out(out + (size_t)kept * per, d + o_kept, (size_t)n * per * sizeof(double));
    if (trial_index) scratch.out(trial_index + kept, d + o_trial, (size_t)n * sizeof(int));
    kept += n;
    done += set;
    const double pass = (double)std::max(kept, 1) / done;
    set = (int)std::min<double>(std::min<double>(ntrial - done, (double)cap),
                                std::max(4096.0, 1.25 * (max_keep - kept) / pass));
  }
  return kept;
}

}  // namespace cdk
