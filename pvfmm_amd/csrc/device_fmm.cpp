// Builds the per-tree device plan and runs one evaluation (the reference's RunFMM,
// include/fmm_tree.txx:237-738, with the list setups of include/fmm_pts.txx:2275-5737
// expressed as flat index arrays).
#include "device_fmm.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <string>
#include <unordered_map>

#include "device_ops.hpp"
#include "kernels.hpp"

namespace pvfmm_amd {

void throw_device_error(hipError_t e, const char* file, int line) {
  throw Error(e == hipErrorOutOfMemory ? kErrOutOfMemory : kErrDevice,
              std::string("HIP error '") + hipGetErrorString(e) + "' at " + file + ":" + std::to_string(line));
}

static std::atomic<uint64_t> g_plan_generation{0};
DevicePlanBase::DevicePlanBase() : generation(++g_plan_generation) {}

const char* phase_name(int p) {
  static const char* names[] = {"Gather", "S2U-P2P", "S2U-GEMM", "U2U", "X-List", "V-List:FFT", "V-List:Hadamard",
                                "V-List:IFFT", "D2D", "D2T-GEMM", "D2T+W-List", "U-List", "Scatter"};
  return (p >= 0 && p < kPhaseCount) ? names[p] : "?";
}

namespace {

// LDS pool slots of the V-list tiles' staged partners for the fp16 kernel (FP32 scalar
// kernels), which keeps one pool of `pool` staged entries across the run of tiles a block
// handles: a partner of tile k that tile k-1 also lists keeps its slot, and only the others
// (the delta) are read and staged, into slots that no partner of tile k-1 holds, while tile
// k-1 is computed.  A block's first tile stages its whole union into the same slots.
// Among the free slots, a new partner takes one by greedy colouring, most-read partners
// first: the 16 lanes that read one staged entry each (the 16 targets of a group at one
// offset) are served together, and slot s lands in LDS bank group 7s mod 16, so the slots of
// the partners a group reads at one offset should differ mod 16.  Output: kslot[u] the slot of
// union entry u, and per tile k the delta dent[d0[k] .. d0[k+1]) as (source slot << 9 | slot).
static void assign_pool_slots(int n_off, int pool, int n_s, const std::vector<int32_t>& t0, const std::vector<int32_t>& u0,
                              const std::vector<int32_t>& usrc, const std::vector<int32_t>& partner,
                              std::vector<int32_t>& kslot, std::vector<int32_t>& d0, std::vector<int32_t>& dent) {
  constexpr int G = 16;
  const int n_tiles = (int)t0.size() - 1;
  kslot.assign(usrc.size(), -1);
  d0.assign(1, 0);
  dent.clear();
  std::vector<int32_t> slot_of(std::max(1, n_s), -1);  // slots of the partners of the last tile
  std::vector<int32_t> loc(std::max(1, n_s), -1);      // local index in the current tile
  std::vector<char> busy(pool);
  for (int k = 0; k < n_tiles; k++) {
    const int nu = u0[k + 1] - u0[k];
    for (int u = u0[k]; u < u0[k + 1]; u++) loc[usrc[u]] = u - u0[k];
    std::fill(busy.begin(), busy.end(), 0);
    if (k > 0)
      for (int u = u0[k - 1]; u < u0[k]; u++) {
        const int32_t sl = usrc[u];
        busy[slot_of[sl]] = 1;
        if (loc[sl] < 0) slot_of[sl] = -1;  // dropped: a later listing starts a new run
      }
    // groups of local indices read together, as (group, offset) of the tile
    std::vector<std::vector<int>> grp, memb(nu);
    for (int g = 0; g < 4; g++)
      for (int o = 0; o < n_off; o++) {
        std::vector<int> m;
        for (int r = 0; r < 16; r++) {
          const int t = t0[k] + 16 * g + r;
          if (t >= t0[k + 1]) break;
          const int32_t sl = partner[(size_t)t * n_off + o];
          if (sl >= 0) m.push_back(loc[sl]);
        }
        std::sort(m.begin(), m.end());
        m.erase(std::unique(m.begin(), m.end()), m.end());
        if (m.size() < 2) continue;
        for (int li : m) memb[li].push_back((int)grp.size());
        grp.push_back(std::move(m));
      }
    std::vector<int> col(nu, -1), order;
    for (int li = 0; li < nu; li++) {
      const int32_t sl = usrc[u0[k] + li];
      if (slot_of[sl] >= 0) col[li] = slot_of[sl] % G;  // kept
      else order.push_back(li);
    }
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return memb[x].size() > memb[y].size(); });
    for (int li : order) {
      int bad[G] = {0};
      for (int gi : memb[li])
        for (int lj : grp[gi])
          if (col[lj] >= 0) bad[col[lj]]++;
      int best = -1, best_slot = -1;
      for (int c = 0; c < G; c++) {
        int s = c;
        while (s < pool && busy[s]) s += G;
        if (s >= pool) continue;
        if (best < 0 || bad[c] < bad[best] || (bad[c] == bad[best] && s < best_slot)) { best = c; best_slot = s; }
      }
      if (best < 0) throw Error(kErrInternal, "V-list tiles exceed the staging pool");
      const int32_t sl = usrc[u0[k] + li];
      busy[best_slot] = 1;
      slot_of[sl] = best_slot;
      col[li] = best;
      dent.push_back((sl << 9) | best_slot);
    }
    for (int u = u0[k]; u < u0[k + 1]; u++) {
      kslot[u] = slot_of[usrc[u]];
      loc[usrc[u]] = -1;
    }
    d0.push_back((int32_t)dent.size());
  }
  // replay the staging as the kernel does it: each tile's delta goes to slots its predecessor
  // does not read, after which every slot of the tile's table holds the listed source
  std::vector<int32_t> held(pool, -1);
  for (int k = 0; k < n_tiles; k++) {
    if (k > 0) std::fill(busy.begin(), busy.end(), 0);
    if (k > 0)
      for (int u = u0[k - 1]; u < u0[k]; u++) busy[kslot[u]] = 1;
    for (int d = d0[k]; d < d0[k + 1]; d++) {
      const int s = dent[d] & 511;
      if (s >= pool || (k > 0 && busy[s])) throw Error(kErrInternal, "V-list pool slot overwritten while in use");
      held[s] = dent[d] >> 9;
    }
    for (int u = u0[k]; u < u0[k + 1]; u++)
      if (kslot[u] < 0 || kslot[u] >= pool || held[kslot[u]] != usrc[u])
        throw Error(kErrInternal, "V-list pool slot does not hold its partner");
  }
}

template <typename Real>
class DevicePlan final : public DevicePlanBase {
 public:
  DevicePlan(const Octree& T, const Operators& O, std::shared_ptr<DeviceOps<Real>> ops, const double* src_xyz,
             const double* trg_xyz, int n_vec, hipStream_t s)
      : O_(O), ops_(std::move(ops)), st_(s) {
    n_vec_max = std::max(1, n_vec);
    build(T, src_xyz, trg_xyz);
  }

  hipStream_t stream() const override { return st_; }
  bool is_fp32() const override { return sizeof(Real) == 4; }

  void evaluate(const double* d_den, double* d_out, int n_vec, double den_scale, double out_scale) override {
    if (n_vec < 1) throw Error(kErrInvalidArgument, "n_vec must be >= 1");
    // passes of up to n_vec_max vectors: they share the pair geometry of every P2P and run as
    // the rows of one GEMM per up/down step
    for (int v = 0; v < n_vec; v += nvb_)
      evaluate_one(d_den + (int64_t)v * k0_ * n_src_, d_out + (int64_t)v * k1_ * n_trg_, den_scale, out_scale,
                   std::min(nvb_, n_vec - v));
  }

  void evaluate_slots(const double* const* den_slot, double* const* out_slot) override {
    evaluate_one(nullptr, nullptr, 1.0, 1.0, 1, den_slot, out_slot);
  }

  int64_t device_bytes() const override { return device_bytes_ + ops_->bytes(); }

  Tuning autotune(const double* d_den, double* d_out, int n_vec) override {
    if (n_vec < 1 || n_vec > nvb_) throw Error(kErrInvalidArgument, "autotune takes 1 to n_vec_max density vectors");
    const bool was = timing_;
    timing_ = true;
    // fastest per-phase times over a few evaluations with the current tuning
    auto measure = [&]() {
      std::vector<double> best(kPhaseCount, 1e300);
      for (int r = 0; r < 3; r++) {
        evaluate_one(d_den, d_out, 1.0, 1.0, n_vec);
        for (int p = 0; p < kPhaseCount; p++) best[p] = std::min(best[p], phase_ms[p]);
      }
      return best;
    };
    auto pick = [&](int& knob, std::initializer_list<int> cands, std::initializer_list<int> phases) {
      int best_v = knob;
      double best_t = 1e300;
      for (int v : cands) {
        knob = v;
        const std::vector<double> ph = measure();
        double t = 0;
        for (int p : phases) t += ph[p];
        if (t < best_t) { best_t = t; best_v = v; }
      }
      knob = best_v;
    };
    try {
      if (sizeof(Real) == 4 && e0_ == 1 && vt_.n > 0) {
        pick(tuning.hadamard_tpb, {4, 8, 16, 32, 64}, {kPhHadamard});
      }
      pick(tuning.gemm_split_blocks, {0, 256, 512, 1024, 2048}, {kPhS2UGemm, kPhU2U, kPhD2D, kPhD2TGemm});
    } catch (...) {
      timing_ = was;
      throw;
    }
    timing_ = was;
    return tuning;
  }

 private:
  using K = DeviceKernels<Real>;
  const Operators& O_;
  std::shared_ptr<DeviceOps<Real>> ops_;  // the operators on the device, shared with other trees
  hipStream_t st_;
  int64_t n_src_ = 0, n_trg_ = 0;
  int k0_ = 1, k1_ = 1, e0_ = 1, e1_ = 1, K0_ = 0, K1_ = 0, ns_ = 0, m_ = 0, M_dim_ = 0;
  int n_nodes_ = 0, max_depth_ = 0;
  int bndry_ = 0;     // boundary type of the tree (0 free space, 1-3 periodic)
  const Real* bc_ = nullptr;  // periodic boundary operator (K0_ x K1_)
  bool vol_ = false;  // PXYZ with a kernel carrying the analytic volume potential
  DBuf<double> txa_;  // target coordinates in sorted order (SoA), for the volume-potential correction

  // tree arrays (periodic trees append virtual image nodes: a source node's point range and size
  // with its centre moved by whole periods)
  DBuf<double> center_;
  DBuf<float> node_size_;
  DBuf<int32_t> src_begin_, src_end_, trg_begin_, trg_end_;
  DBuf<int64_t> src_perm_, trg_perm_;
  DBuf<Real> sx_, tx_, sden_;
  DBuf<double> sx64_, tx64_;  // FP64 leaf-local coordinates for the U list
  DBuf<double> tval_;
  // expansions: eq_ = [up (n_nodes x K0) | L2T equivalent rows (n_l2t x K0)]
  DBuf<Real> eq_, dn_, chk_;
  DBuf<Real> ctmp_;
  // U2U / D2D through the check-to-equivalent rank (DeviceOps::u2ur, d2dr) at levels of at least
  // kFactorRows parents (a smaller level costs less as one GEMM than as two launches);
  // lvl_seq_ = 0, 1, ... (rows of ctmp_)
  static constexpr int kFactorRows = 256;
  static constexpr int kVListSlots = 4096;
  static constexpr int64_t kVListBytes = int64_t(1) << 31;
  DBuf<int32_t> lvl_seq_;
  // the fp16 Hadamard kernels (FP32): the spectrum bound of each slot of X (or, in the adjoint,
  // of Y) and the scale of each run of tiles
  DBuf<float> vbound_, vrscale_;
  bool split_ = false;
  // split-K partial tiles of the small coarse-level GEMMs: room for 4 of the largest output, at most 2^25
  DBuf<Real> gemm_work_;
  int64_t gemm_work_elems_ = 0;
  int nvb_ = 1;  // density vectors per evaluation pass (buffers hold this many)
  int64_t eq_vs_ = 0, dn_vs_ = 0, chk_vs_ = 0, ctmp_vs_ = 0;  // per-vector strides
  int ru_ = 0, rd_ = 0;
  // The coarsest level whose upward equivalent densities anything reads (V or W list, boundary
  // operator), and whose downward check potentials anything writes: U2U and D2D stop there (in
  // free space the two coarsest levels have no V or W list and their translations were zeros or
  // unread; 20 of 250 us at 4099 points)
  int up_min_ = 0, dn_min_ = 0;
  // S2M
  DBuf<int32_t> s2m_node_, s2m_ptr_, s2m_items_, s2m_orow_;
  DBuf<Real> s2m_alpha_;
  int n_s2m_ = 0;
  // M2M / L2L per level
  struct LevelRows { int n = 0; DBuf<int32_t> ra, rc; };
  std::vector<std::unique_ptr<LevelRows>> m2m_, l2l_;
  // X list
  DBuf<int32_t> x_node_, x_ptr_, x_items_, x_orow_;
  int n_x_ = 0;
  // V list
  DBuf<int32_t> v_src_fc_, v_trg_fc_, v_offsets_;
  DBuf<Real> v_src_scal_, v_trg_scal_, X_, Y_;
  // density vectors of one V-list pass: the spectra buffers hold that many, with these strides
  int vlist_nv_ = 1;
  int64_t x_vs_ = 0, y_vs_ = 0, bound_vs_ = 0;
  int n_vsrc_ = 0, n_vtrg_ = 0, n_off_ = 0;

  // V-list target tiles for the LDS-staged Hadamard
  struct TileSet {
    DBuf<int32_t> t0, u0, usrc;
    DBuf<uint16_t> uidx;
    DBuf<uint32_t> gmask;
    DBuf<int32_t> d0, dent;  // FP32 scalar kernel: per tile, the partners new since the previous tile
    int n = 0;
    int64_t partners = 0, max_partners = 0, staged_delta = 0;
  };
  TileSet vt_;
  // rows of A (K) -> rank R -> rows of C (N): one launch where that is the faster form, else two
  // products with the intermediate rows seq of ctmp_
  void pair(const typename DeviceOps<Real>::PackedPair& p, const DBuf<Real>& B1, const DBuf<Real>& B2, int M, int K, int R, int N,
            const Real* A, const int32_t* ra, const Real* alpha1, const int32_t* seq, Real* C, const int32_t* rc,
            const Real* alpha2, bool accumulate, int nv, int64_t avs, int64_t cvs) {
    if (p.use && DeviceKernels<Real>::gemm_pair_pays(K, (int64_t)M * nv)) {
      DeviceKernels<Real>::gemm_pair(st_, M, K, R, N, A, ra, K, p.B1.p, alpha1, p.B2.p, C, rc, N, alpha2, accumulate, nv, avs, cvs);
      return;
    }
    const int sp = tuning.gemm_split_blocks;
    DeviceKernels<Real>::gemm_rows(st_, M, R, K, A, ra, K, B1.p, ctmp_.p, seq, R, alpha1, false, gemm_work_.p, gemm_work_elems_, sp,
                                   nv, avs, ctmp_vs_);
    DeviceKernels<Real>::gemm_rows(st_, M, N, R, ctmp_.p, seq, R, B2.p, C, rc, N, alpha2, accumulate, gemm_work_.p,
                                   gemm_work_elems_, sp, nv, ctmp_vs_, cvs);
  }
  // operands of the fp16 Hadamard with run scales in `rs` (kept until the launch returns)
  HadamardParts hp_;
  const HadamardParts& hparts(DBuf<float>& rs) {
    hp_.Vh = ops_->Vh.p;
    hp_.tinv = ops_->vtinv.p;
    hp_.bound = vbound_.p;
    hp_.run_scale = rs.p;
    hp_.run_scale_cap = (int)rs.n;
    hp_.bound_vs = bound_vs_;
    return hp_;
  }

  // Tiles of consecutive target slots: at most 64 targets, at most umax distinct partners
  // (greedy in slot order, which is Morton order within a level).  partner[t * n_off + o] is
  // the source slot of target slot t at offset o, or -1.  For the FP32 scalar kernel (LDS pool
  // of assign_pool_slots) a tile's partners together with the previous tile's must also fit
  // the pool, and usrc holds each tile's union as (source slot << 9 | pool slot).
  void build_tiles(const std::vector<int32_t>& v_partner, int n_t, int n_s, TileSet& ts, int64_t* total) {
    const int umax = K::hadamard_union_max(e0_);
    const bool pair_layout = std::is_same<Real, float>::value && e0_ == 1 && e1_ == 1;
    const int pool = pair_layout ? K::hadamard_pool_max() : (1 << 30);
    std::vector<int32_t> t0{0}, u0{0}, usrc;
    std::vector<uint16_t> uidx;
    std::vector<int32_t> pos(std::max(1, n_s), -1);
    std::vector<char> in_prev(std::max(1, n_s), 0);  // partner of the last closed tile
    std::vector<int32_t> cur, prev;  // distinct partners of the open tile and of the last closed one
    int cur_new = 0;                 // partners of the open tile that the last closed one lacks
    auto close_tile = [&](int t_end) {
      for (int32_t sl : cur) pos[sl] = -1;
      usrc.insert(usrc.end(), cur.begin(), cur.end());
      for (int32_t sl : prev) in_prev[sl] = 0;
      prev.swap(cur);
      for (int32_t sl : prev) in_prev[sl] = 1;
      cur.clear();
      cur_new = 0;
      t0.push_back(t_end);
      u0.push_back((int32_t)usrc.size());
    };
    // first pass: tile boundaries and union lists
    for (int t = 0; t < n_t; t++) {
      int add = 0, add_new = 0;
      for (int k = 0; k < n_off_; k++) {
        const int32_t sl = v_partner[(size_t)t * n_off_ + k];
        if (sl >= 0 && pos[sl] < 0) { pos[sl] = -2; add++; add_new += in_prev[sl] ? 0 : 1; }  // provisional mark
      }
      for (int k = 0; k < n_off_; k++) {
        const int32_t sl = v_partner[(size_t)t * n_off_ + k];
        if (sl >= 0 && pos[sl] == -2) pos[sl] = -1;
      }
      if (t > t0.back() && (t - t0.back() == 64 || (int)cur.size() + add > umax ||
                            (int64_t)prev.size() + cur_new + add_new > pool))
        close_tile(t);
      for (int k = 0; k < n_off_; k++) {
        const int32_t sl = v_partner[(size_t)t * n_off_ + k];
        if (sl >= 0 && pos[sl] < 0) {
          pos[sl] = (int32_t)cur.size();
          cur.push_back(sl);
          cur_new += in_prev[sl] ? 0 : 1;
        }
      }
    }
    if (n_t > t0.back()) close_tile(n_t);
    const int n_tiles = (int)t0.size() - 1;
    // a missing partner points at the staging area's zero entry (index umax, or the pool size
    // for the FP32 scalar kernel).  The FP32 scalar kernel reads its table as [k][group]
    // [o / 16][o % 2][row][(o / 2) % 8] (pairs o / 2 padded to 16), the others as
    // [k][o][row][group].
    const size_t per_tile = pair_layout ? (size_t)4 * 16 * 2 * 16 : (size_t)64 * n_off_;
    if (pair_layout && n_off_ > 32) throw Error(kErrInternal, "V-list offsets exceed the pair table");
    if (pair_layout && (pool + 1 > 511 || (int64_t)n_s >= (int64_t(1) << 22)))
      throw Error(kErrInternal, "V-list staging pool or source slots exceed the packed entry");
    std::vector<int32_t> kslot, d0, dent;
    if (pair_layout) assign_pool_slots(n_off_, pool, n_s, t0, u0, usrc, v_partner, kslot, d0, dent);
    uidx.assign((size_t)n_tiles * per_tile, (uint16_t)(pair_layout ? pool : umax));
    std::vector<uint32_t> gmask((size_t)n_tiles * 4, 0u);  // offsets present per 16-target group
    for (int k = 0; k < n_tiles; k++) {
      for (int u = u0[k]; u < u0[k + 1]; u++) pos[usrc[u]] = pair_layout ? kslot[u] : u - u0[k];
      for (int t = t0[k]; t < t0[k + 1]; t++)
        for (int o = 0; o < n_off_; o++) {
          const int32_t sl = v_partner[(size_t)t * n_off_ + o];
          const int tt = t - t0[k];  // target tt = 16 * group + row of the MFMA tiles
          if (sl >= 0) {
            const size_t at = pair_layout ? (size_t)k * per_tile +
                                                (((((size_t)(tt >> 4) * 2 + (o >> 4)) * 2 + (o & 1)) * 16 + (tt & 15)) * 8 +
                                                 ((o >> 1) & 7))
                                          : (((size_t)k * n_off_ + o) * 16 + (tt & 15)) * 4 + (tt >> 4);
            uidx[at] = (uint16_t)pos[sl];
            gmask[(size_t)k * 4 + (tt >> 4)] |= 1u << o;
          }
        }
      for (int u = u0[k]; u < u0[k + 1]; u++) pos[usrc[u]] = -1;
      if (u0[k + 1] - u0[k] > umax || t0[k + 1] - t0[k] > 64)
        throw Error(kErrInternal, "V-list tile exceeds its staging capacity");
      ts.max_partners = std::max<int64_t>(ts.max_partners, u0[k + 1] - u0[k]);
    }
    ts.n = n_tiles;
    ts.partners = (int64_t)usrc.size();
    if (pair_layout) {
      for (size_t u = 0; u < usrc.size(); u++) usrc[u] = (usrc[u] << 9) | kslot[u];
      ts.staged_delta = (int64_t)dent.size();
      // one readable entry past each list's end (source 0 into the unread trash slot): the
      // kernel reads ahead branch-free
      dent.push_back(pool + 1);
      usrc.push_back(pool + 1);
      ts.d0.upload(d0, total);
      ts.dent.upload(dent, total);
    } else {
      ts.staged_delta = ts.partners;
      usrc.push_back(0);  // one readable slot past the end: the kernels read ahead branch-free
    }
    ts.t0.upload(t0, total); ts.u0.upload(u0, total); ts.usrc.upload(usrc, total); ts.uidx.upload(uidx, total);
    ts.gmask.upload(gmask, total);
  }
  // L2T
  DBuf<int32_t> l2t_ra_, l2t_rc_, l2t_seq_;
  DBuf<Real> l2t_alpha_;
  int n_l2t_ = 0;
  // target leaves: far field and U list
  DBuf<int32_t> t_leaf_, far_ptr_, far_node_, u_ptr_, u_items_;
  DBuf<int64_t> far_den_;
  DBuf<double> far_rad_;
  // far rows with much more work than most, split over blocks (FarSplit)
  DBuf<int32_t> fs_row_, fs_begin_, fs_end_, fs_rows_, fs_ptr_;
  DBuf<int64_t> fs_part_;
  DBuf<double> fs_sums_;
  FarSplit far_split_;
  int n_tleaf_ = 0;
  std::vector<hipEvent_t> ev_;
  std::vector<hipEvent_t> vev_;  // per-vector V-list sub-phase events (timing of multi-vector passes)

 public:
  ~DevicePlan() override {
    for (hipEvent_t e : ev_) (void)hipEventDestroy(e);
    for (hipEvent_t e : vev_) (void)hipEventDestroy(e);
  }

 private:
  void mark(int phase) {
    if (timing_) HIP_CHECK(hipEventRecord(ev_[phase], st_));
  }
  void ensure_vlist_events(int nv) {
    while ((int)vev_.size() < 4 * nv) {
      hipEvent_t e = nullptr;
      HIP_CHECK(hipEventCreate(&e));
      vev_.push_back(e);
    }
  }

  void build(const Octree& T, const double* src_xyz, const double* trg_xyz) {
    int64_t total = 0;
    const KernelInfo& ki = O_.ker;
    k0_ = ki.k0; k1_ = ki.k1; e0_ = ki.e0; e1_ = ki.e1;
    ns_ = O_.ns; m_ = O_.m; K0_ = O_.K0(); K1_ = O_.K1(); M_dim_ = ops_->grid.M;
    n_src_ = T.src.n; n_trg_ = T.trg.n;
    n_nodes_ = T.n_nodes();
    max_depth_ = T.max_depth;
    if (n_src_ >= (1ll << 31) || n_trg_ >= (1ll << 31)) throw Error(kErrUnsupported, "more than 2^31 points");
    const int N = n_nodes_;
    bndry_ = T.bndry;

    // ---- periodic images: every (source node, shift) that a U, W or X list of a target node
    // reaches across the boundary becomes a virtual node N + j
    std::unordered_map<int64_t, int32_t> img_of;
    std::vector<std::pair<int32_t, int>> imgs;  // (source node, shift code (sx+1) + 3(sy+1) + 9(sz+1))
    auto img = [&](int32_t t, int type, int k, int32_t s) -> int32_t {
      if (bndry_ == kFreeSpace) return s;
      int sh[3];
      image_shift(T, t, s, type, k, sh);
      const int code = (sh[0] + 1) + 3 * (sh[1] + 1) + 9 * (sh[2] + 1);
      if (code == 13) return s;
      const int64_t key = (int64_t)s * 27 + code;
      auto it = img_of.find(key);
      if (it != img_of.end()) return it->second;
      const int32_t v = N + (int32_t)imgs.size();
      img_of.emplace(key, v);
      imgs.emplace_back(s, code);
      return v;
    };
    if (bndry_ != kFreeSpace)
      for (int t = 0; t < N; t++) {
        if (T.pt_cnt1(t) == 0) continue;
        for (int type : {kU0, kU1, kU2, kW, kX}) {
          const int nl = T.list_count(type);
          for (int k = 0; k < nl; k++) {
            const int32_t s = T.lists[type][(size_t)t * nl + k];
            if (s >= 0) (void)img(t, type, k, s);
          }
        }
      }
    const int NV = N + (int)imgs.size();

    // ---- node arrays
    std::vector<double> center(3 * (size_t)NV);
    std::vector<float> nsz(NV);
    std::vector<int32_t> sb(NV), se(NV), tb(NV, 0), te(NV, 0);
    for (int i = 0; i < N; i++) {
      double c[3];
      T.corner(i, c);
      double s = T.size(i);
      for (int d = 0; d < 3; d++) center[3 * i + d] = c[d] + 0.5 * s;
      nsz[i] = (float)s;
      sb[i] = (int32_t)T.src_begin[i]; se[i] = (int32_t)T.src_end[i];
      tb[i] = (int32_t)T.trg_begin[i]; te[i] = (int32_t)T.trg_end[i];
    }
    for (size_t j = 0; j < imgs.size(); j++) {
      const int32_t s = imgs[j].first, v = N + (int32_t)j, code = imgs[j].second;
      const int sh[3] = {code % 3 - 1, (code / 3) % 3 - 1, code / 9 - 1};
      for (int d = 0; d < 3; d++) center[3 * (size_t)v + d] = center[3 * (size_t)s + d] + sh[d];
      nsz[v] = nsz[s];
      sb[v] = sb[s]; se[v] = se[s];
    }
    center_.upload(center, &total);
    node_size_.upload(nsz, &total);
    src_begin_.upload(sb, &total); src_end_.upload(se, &total);
    trg_begin_.upload(tb, &total); trg_end_.upload(te, &total);
    h_.center = center; h_.nsz = nsz; h_.sb = sb; h_.se = se; h_.tb = tb; h_.te = te; h_.imgs = imgs;
    src_perm_.upload(T.src.perm, &total);
    trg_perm_.upload(T.trg.perm, &total);

    // ---- leaf-local coordinates (x - leaf centre), SoA
    std::vector<double> sx(3 * (size_t)n_src_), tx(3 * (size_t)n_trg_);
    for (int i = 0; i < N; i++) {
      if (!T.is_leaf(i)) continue;
      for (int64_t k = T.src_begin[i]; k < T.src_end[i]; k++)
        for (int d = 0; d < 3; d++) sx[d * n_src_ + k] = src_xyz[3 * T.src.perm[k] + d] - center[3 * i + d];
      for (int64_t k = T.trg_begin[i]; k < T.trg_end[i]; k++)
        for (int d = 0; d < 3; d++) tx[d * n_trg_ + k] = trg_xyz[3 * T.trg.perm[k] + d] - center[3 * i + d];
    }
    sx64_.upload(sx, &total);
    tx64_.upload(tx, &total);
    sx_.upload(std::vector<Real>(sx.begin(), sx.end()), &total);
    tx_.upload(std::vector<Real>(tx.begin(), tx.end()), &total);
    // per-vector buffers hold n_vec_max density vectors, one after another
    nvb_ = n_vec_max;
    sden_.alloc((int64_t)k0_ * n_src_ * nvb_, &total);
    tval_.alloc((int64_t)k1_ * n_trg_ * nvb_, &total);

    ru_ = ops_->ru;
    rd_ = ops_->rd;
    split_ = ops_->split;

    const double ts = ki.trg_scal + ki.src_scal;
    // ---- S2M rows: leaves holding sources (Source2UpSetup, include/fmm_pts.txx:2287-2290)
    std::vector<int32_t> s2m_node, s2m_ptr{0}, s2m_items, s2m_orow;
    std::vector<Real> s2m_alpha;
    std::vector<int32_t> l2t_ra, l2t_rc;
    std::vector<Real> l2t_alpha;
    int64_t s2m_pairs = 0;
    for (int i = 0; i < N; i++)
      if (T.is_leaf(i) && T.pt_cnt0(i) > 0) {
        s2m_orow.push_back((int32_t)s2m_node.size());
        s2m_node.push_back(i);
        s2m_items.push_back(i);
        s2m_ptr.push_back((int32_t)s2m_items.size());
        s2m_alpha.push_back((Real)std::pow(2.0, -ts * T.depth[i]));
        s2m_pairs += T.pt_cnt0(i) * ns_;
      }
    n_s2m_ = (int)s2m_node.size();
    h_.s2m_node = s2m_node;
    s2m_node_.upload(s2m_node, &total); s2m_ptr_.upload(s2m_ptr, &total); s2m_items_.upload(s2m_items, &total);
    s2m_orow_.upload(s2m_orow, &total); s2m_alpha_.upload(s2m_alpha, &total);
    chk_vs_ = (int64_t)std::max(1, n_s2m_) * K1_;
    chk_.alloc(chk_vs_ * nvb_, &total);

    // ---- target leaves and L2T rows (Down2TargetSetup, include/fmm_pts.txx:5427-5442)
    std::vector<int32_t> tleaf, l2t_seq;
    for (int i = 0; i < N; i++)
      if (T.is_leaf(i) && T.pt_cnt1(i) > 0) {
        l2t_seq.push_back((int32_t)l2t_ra.size());
        l2t_ra.push_back(i);
        l2t_rc.push_back(N + (int32_t)tleaf.size());  // rows after the up block of eq_
        l2t_alpha.push_back((Real)std::pow(2.0, -ts * T.depth[i]));
        tleaf.push_back(i);
      }
    n_l2t_ = n_tleaf_ = (int)tleaf.size();
    l2t_ra_.upload(l2t_ra, &total); l2t_rc_.upload(l2t_rc, &total); l2t_alpha_.upload(l2t_alpha, &total);
    l2t_seq_.upload(l2t_seq, &total);
    // ctmp_ rows: the check-to-equivalent GEMMs' leaves, and the parents of one level of the
    // rank-factored U2U / D2D
    int max_level_rows = 0;
    for (int l = 0; l <= max_depth_; l++) {
      int na = 0, nb = 0;
      for (int i = T.level_begin[l]; i < T.level_begin[l + 1]; i++) {
        if (T.is_leaf(i)) continue;
        na += T.pt_cnt0(i) > 0;
        nb += T.pt_cnt1(i) > 0;
      }
      max_level_rows = std::max(max_level_rows, std::max(na, nb));
    }
    {
      std::vector<int32_t> seq(std::max(1, max_level_rows));
      for (size_t i = 0; i < seq.size(); i++) seq[i] = (int32_t)i;
      lvl_seq_.upload(seq, &total);
    }
    ctmp_vs_ = (int64_t)std::max(1, std::max(std::max(n_s2m_, n_l2t_), max_level_rows)) * std::max(1, std::max(ru_, rd_));
    ctmp_.alloc(ctmp_vs_ * nvb_, &total);
    t_leaf_.upload(tleaf, &total);
    eq_vs_ = (int64_t)(N + n_l2t_) * K0_;
    dn_vs_ = (int64_t)N * K1_;
    auto words = [](int64_t count) { return (count + 3) / 4 * 4; };  // whole 16-byte words (begin)
    eq_.alloc(words(eq_vs_ * nvb_), &total);
    dn_.alloc(words(dn_vs_ * nvb_), &total);

    // ---- M2M / L2L rows per level
    m2m_.clear(); l2l_.clear();
    int64_t m2m_rows = 0, l2l_rows = 0;
    for (int l = 0; l <= max_depth_; l++) {
      auto a = std::make_unique<LevelRows>(), b = std::make_unique<LevelRows>();
      std::vector<int32_t> ra, rc, ra2, rc2;
      for (int i = T.level_begin[l]; i < T.level_begin[l + 1]; i++) {
        if (T.is_leaf(i)) continue;
        if (T.pt_cnt0(i) > 0) { ra.push_back(T.first_child[i]); rc.push_back(i); }  // Up2UpSetup 2618-2619
        if (T.pt_cnt1(i) > 0) { ra2.push_back(i); rc2.push_back(T.first_child[i]); }  // Down2DownSetup 3777-3778
      }
      a->n = (int)ra.size(); a->ra.upload(ra, &total); a->rc.upload(rc, &total);
      b->n = (int)ra2.size(); b->ra.upload(ra2, &total); b->rc.upload(rc2, &total);
      m2m_rows += a->n; l2l_rows += b->n;
      m2m_.push_back(std::move(a)); l2l_.push_back(std::move(b));
    }
    {
      int64_t out = std::max((int64_t)n_s2m_ * std::max(ru_, K0_), (int64_t)n_l2t_ * std::max(rd_, K0_));
      for (auto& L : m2m_) out = std::max(out, (int64_t)L->n * K0_);
      for (auto& L : l2l_) out = std::max(out, (int64_t)L->n * 8 * K1_);
      gemm_work_elems_ = std::min<int64_t>(int64_t(1) << 25, std::max<int64_t>(1, 4 * out * nvb_));
      gemm_work_.alloc(gemm_work_elems_, &total);
    }

    const int nl_x = T.list_count(kX), nl_w = T.list_count(kW);
    // ---- X list S2L (X_ListSetup, include/fmm_pts.txx:4444-4743)
    std::vector<int32_t> x_node, x_ptr{0}, x_items, x_orow;
    for (int i = 0; i < N; i++) {
      if (T.pt_cnt1(i) == 0) continue;
      if (T.is_leaf(i) && T.pt_cnt1(i) <= ns_) continue;  // handled in the U list
      int cnt = 0;
      for (int k = 0; k < nl_x; k++) {
        int32_t s = T.lists[kX][(size_t)i * nl_x + k];
        if (s >= 0 && T.is_leaf(s) && T.pt_cnt0(s) > 0) { x_items.push_back(img(i, kX, k, s)); cnt++; }
      }
      if (!cnt) continue;
      x_node.push_back(i); x_orow.push_back(i);
      x_ptr.push_back((int32_t)x_items.size());
    }
    n_x_ = (int)x_node.size();
    x_node_.upload(x_node, &total); x_ptr_.upload(x_ptr, &total); x_items_.upload(x_items, &total); x_orow_.upload(x_orow, &total);
    h_.x_node = x_node; h_.x_ptr = x_ptr; h_.x_items = x_items;

    // ---- V list (V_ListSetup, include/fmm_pts.txx:3346-3595): parents holding sources / targets
    std::vector<int32_t> slot_of(N, -1), v_src_fc, v_trg_fc, v_partner;
    std::vector<Real> v_src_scal, v_trg_scal;
    for (int i = 0; i < N; i++)
      if (!T.is_leaf(i) && T.pt_cnt0(i) > 0) {
        slot_of[i] = (int32_t)v_src_fc.size();
        v_src_fc.push_back(T.first_child[i]);
        v_src_scal.push_back((Real)std::pow(2.0, ki.src_scal * (T.depth[i] + 1)));
        h_.vsrc_depth.push_back(T.depth[i]);
      }
    std::vector<int32_t> offs(O_.v1_offsets.begin(), O_.v1_offsets.end());
    n_off_ = (int)offs.size();
    int64_t v_pairs = 0;
    const int nl_v1 = T.list_count(kV1);
    const RelTable& v1t = rel_table(kV1);
    for (int i = 0; i < N; i++) {
      if (T.is_leaf(i) || T.pt_cnt1(i) == 0) continue;
      std::vector<int32_t> row(n_off_, -1);
      int cnt = 0;
      for (int k = 0; k < nl_v1; k++) {
        int32_t s = T.lists[kV1][(size_t)i * nl_v1 + k];
        if (s < 0 || T.pt_cnt0(s) == 0) continue;
        const auto& r = v1t.rel[k];
        int R = (r[0] + 1) + 3 * (r[1] + 1) + 9 * (r[2] + 1);
        int oi = (int)(std::find(offs.begin(), offs.end(), R) - offs.begin());
        row[oi] = slot_of[s];
        cnt++;
      }
      if (!cnt) continue;
      v_pairs += cnt;
      v_trg_fc.push_back(T.first_child[i]);
      v_trg_scal.push_back((Real)std::pow(2.0, ki.trg_scal * (T.depth[i] + 1)));
      h_.vtrg_depth.push_back(T.depth[i]);
      v_partner.insert(v_partner.end(), row.begin(), row.end());
    }
    n_vsrc_ = (int)v_src_fc.size();
    n_vtrg_ = (int)v_trg_fc.size();
    v_src_fc_.upload(v_src_fc, &total); v_trg_fc_.upload(v_trg_fc, &total);
    v_src_scal_.upload(v_src_scal, &total); v_trg_scal_.upload(v_trg_scal, &total);
    v_offsets_.upload(offs, &total);
    h_.v_partner = v_partner; h_.v_src_fc = v_src_fc; h_.v_trg_fc = v_trg_fc; h_.offs = offs;
    build_tiles(v_partner, n_vtrg_, n_vsrc_, vt_, &total);
    // A V-list pass takes as many vectors as make about kVListSlots source or target parents (a
    // parent is one block of a transform), so that a small tree's pass fills the chip, and whose
    // spectra fit kVListBytes, which many trees may keep side by side; a large tree's takes one,
    // whose spectra alone may be gigabytes.
    x_vs_ = (int64_t)n_vsrc_ * M_dim_ * 16 * e0_;
    y_vs_ = (int64_t)n_vtrg_ * M_dim_ * 16 * e1_;
    vlist_nv_ = std::max(1, std::min(nvb_, kVListSlots / std::max(1, std::max(n_vsrc_, n_vtrg_))));
    vlist_nv_ = (int)std::max<int64_t>(1, std::min<int64_t>(vlist_nv_, kVListBytes / (int64_t)sizeof(Real) / std::max<int64_t>(1, x_vs_ + y_vs_)));
    if (split_) {
      // per slot and component; the adjoint's sources are the target slots
      bound_vs_ = std::max(1, std::max(n_vsrc_ * e0_, n_vtrg_ * e1_));
      vbound_.alloc(bound_vs_ * vlist_nv_, &total);
      vrscale_.alloc((int64_t)2 * std::max(1, vt_.n) * vlist_nv_, &total);
    }
    stats.v_tiles = vt_.n;
    stats.v_tile_partners = vt_.partners;
    stats.v_tile_max_partners = vt_.max_partners;
    stats.v_tile_staged = vt_.staged_delta;
    X_.alloc(x_vs_ * vlist_nv_, &total);
    Y_.alloc(y_vs_ * vlist_nv_, &total);

    up_min_ = dn_min_ = bndry_ != kFreeSpace ? 0 : max_depth_ + 1;
    {
      const int nl_vw = T.list_count(kW);
      std::vector<char> used_src(n_vsrc_, 0);
      for (int32_t sl : v_partner)
        if (sl >= 0) used_src[sl] = 1;
      for (int sl = 0; sl < n_vsrc_; sl++)
        if (used_src[sl]) up_min_ = std::min(up_min_, h_.vsrc_depth[sl] + 1);
      for (int d : h_.vtrg_depth) dn_min_ = std::min(dn_min_, d + 1);
      for (int i : x_node) dn_min_ = std::min(dn_min_, (int)T.depth[i]);
      for (int t : tleaf)
        for (int k = 0; k < nl_vw; k++) {
          const int32_t w = T.lists[kW][(size_t)t * nl_vw + k];
          if (w >= 0) up_min_ = std::min(up_min_, (int)T.depth[w]);
        }
    }

    // ---- far field (L2T own surface + W list M2T) and U list per target leaf
    std::vector<int32_t> far_ptr{0}, far_node, u_ptr{0}, u_items;
    std::vector<int64_t> far_den;
    std::vector<double> far_rad;
    const int nl_u0 = T.list_count(kU0), nl_u1 = T.list_count(kU1), nl_u2 = T.list_count(kU2);
    int64_t u_pairs = 0, far_pairs = 0, u_stream = 0;
    for (int r = 0; r < n_tleaf_; r++) {
      const int t = tleaf[r];
      far_node.push_back(t); far_den.push_back((int64_t)(N + r) * K0_); far_rad.push_back(kRad1);
      for (int k = 0; k < nl_w; k++) {  // W_ListSetup 4910-4913
        int32_t s = T.lists[kW][(size_t)t * nl_w + k];
        if (s < 0 || T.pt_cnt0(s) == 0) continue;
        if (T.is_leaf(s) && T.pt_cnt0(s) <= ns_) continue;
        far_node.push_back(img(t, kW, k, s)); far_den.push_back((int64_t)s * K0_); far_rad.push_back(kRad0);
      }
      far_pairs += (int64_t)(far_node.size() - far_ptr.back()) * ns_ * T.pt_cnt1(t);
      far_ptr.push_back((int32_t)far_node.size());
      auto add = [&](int32_t s, int type, int k) {
        if (s >= 0 && T.is_leaf(s) && T.pt_cnt0(s) > 0) {
          u_items.push_back(img(t, type, k, s));
          u_pairs += T.pt_cnt0(s) * T.pt_cnt1(t);
          u_stream += T.pt_cnt0(s);
        }
      };
      for (int k = 0; k < nl_u0; k++) add(T.lists[kU0][(size_t)t * nl_u0 + k], kU0, k);  // U_ListSetup 5197-5321
      for (int k = 0; k < nl_u1; k++) add(T.lists[kU1][(size_t)t * nl_u1 + k], kU1, k);
      for (int k = 0; k < nl_u2; k++) add(T.lists[kU2][(size_t)t * nl_u2 + k], kU2, k);
      if (T.pt_cnt1(t) <= ns_)
        for (int k = 0; k < nl_x; k++) add(T.lists[kX][(size_t)t * nl_x + k], kX, k);
      for (int k = 0; k < nl_w; k++) {
        int32_t s = T.lists[kW][(size_t)t * nl_w + k];
        if (s >= 0 && T.is_leaf(s) && T.pt_cnt0(s) <= ns_) add(s, kW, k);
      }
      u_ptr.push_back((int32_t)u_items.size());
    }
    far_ptr_.upload(far_ptr, &total); far_node_.upload(far_node, &total); far_den_.upload(far_den, &total);
    far_rad_.upload(far_rad, &total);
    split_far_rows(T, tleaf, far_ptr, &total);
    u_ptr_.upload(u_ptr, &total); u_items_.upload(u_items, &total);
    if (bndry_ != kFreeSpace) {  // FMM_Pts::PeriodicBC and PostProcessing (include/fmm_pts.txx:2641-2657,5740-5774)
      bc_ = ops_->bc(bndry_, false);
      vol_ = bndry_ == kPXYZ && ki.id != 1;
      if (vol_) {
        std::vector<double> xa(3 * (size_t)n_trg_);
        for (int64_t k = 0; k < n_trg_; k++)
          for (int d = 0; d < 3; d++) xa[d * n_trg_ + k] = trg_xyz[3 * T.trg.perm[k] + d];
        txa_.upload(xa, &total);
      }
    }
    h_.tleaf = tleaf; h_.u_ptr = u_ptr; h_.u_items = u_items;
    h_.far_ptr = far_ptr; h_.far_node = far_node; h_.far_rad = far_rad;

    ev_.resize(kPhaseCount + 1);
    for (auto& e : ev_) HIP_CHECK(hipEventCreate(&e));
    phase_ms.assign(kPhaseCount, 0.0);

    stats.n_nodes = N;
    for (int i = 0; i < N; i++) stats.n_leaves += T.is_leaf(i);
    stats.max_depth = max_depth_;
    stats.s2m_rows = n_s2m_; stats.l2t_rows = n_l2t_; stats.m2m_rows = m2m_rows; stats.l2l_rows = l2l_rows;
    stats.x_rows = n_x_; stats.x_items = (int64_t)x_items.size();
    stats.v_src_slots = n_vsrc_; stats.v_trg_slots = n_vtrg_; stats.v_pairs = v_pairs;
    stats.u_rows = n_tleaf_; stats.u_items = (int64_t)u_items.size(); stats.u_pairs = u_pairs;
    stats.u_src_points_streamed = u_stream;
    stats.far_items = (int64_t)far_node.size(); stats.far_pairs = far_pairs; stats.s2m_pairs = s2m_pairs;
    device_bytes_ = total;
  }

  // Splits the far rows of more than kFarRowPairs pairs into segments of about kFarSegPairs, or of
  // one item where that is more (with m = 10 from 67 targets on).  A block of 256 threads does
  // 5,000-20,000 pairs, the mean row of ordinary trees, in 10-30 us; a row of 16 such units would
  // outlast the rest of most launches.  Trees of few large leaves need it most: with rows split
  // above 4 times their mean only, 200,000 points in leaves of up to 3000 (m = 10) took 2.45 ms
  // instead of 0.40.  But there nearly every row with W items is split, and a sum per segment and
  // target was up to 17 times the outputs: where the sums would be more than kFarSums times the
  // outputs (and 2^20 values per vector), the segments are longer.  Segments go first.
  static constexpr int64_t kFarRowPairs = 131072, kFarSegPairs = 32768, kFarSums = 4;
  void split_far_rows(const Octree& T, const std::vector<int32_t>& tleaf, const std::vector<int32_t>& far_ptr, int64_t* total) {
    std::vector<int32_t> row, begin, end, rows, ptr{0};
    std::vector<int64_t> part;
    std::vector<char> heavy(tleaf.size(), 0);
    int64_t sums = 0, seg_pairs = kFarSegPairs;
    auto per_seg = [&](size_t r) {  // items of a segment of row r, 0: the row stays whole
      const int64_t item = (int64_t)T.pt_cnt1(tleaf[r]) * ns_, n = far_ptr[r + 1] - far_ptr[r];
      const int64_t per = std::max<int64_t>(1, seg_pairs / item);
      return n * item <= kFarRowPairs || per >= n ? 0 : (int)per;
    };
    for (;; seg_pairs *= 2) {
      int64_t room = std::max<int64_t>(kFarSums * n_trg_ * k1_, 1 << 20);
      for (size_t r = 0; r < tleaf.size() && room >= 0; r++)
        if (const int per = per_seg(r))
          room -= (far_ptr[r + 1] - far_ptr[r] + per - 1) / per * (int64_t)T.pt_cnt1(tleaf[r]) * k1_;
      if (room >= 0) break;
    }
    for (size_t r = 0; r < tleaf.size(); r++) {
      const int64_t nt = T.pt_cnt1(tleaf[r]);
      const int per = per_seg(r);
      if (per == 0) continue;
      for (int i = far_ptr[r]; i < far_ptr[r + 1]; i += per) {
        row.push_back((int32_t)r);
        begin.push_back(i);
        end.push_back(std::min(far_ptr[r + 1], i + per));
        part.push_back(sums);
        sums += nt * k1_;
      }
      heavy[r] = 1;
      rows.push_back((int32_t)r);
      ptr.push_back((int32_t)row.size());
    }
    if (rows.empty()) return;
    for (size_t r = 0; r < tleaf.size(); r++)
      if (!heavy[r]) {
        row.push_back((int32_t)r);
        begin.push_back(far_ptr[r]);
        end.push_back(far_ptr[r + 1]);
        part.push_back(-1);
      }
    fs_row_.upload(row, total); fs_begin_.upload(begin, total); fs_end_.upload(end, total); fs_part_.upload(part, total);
    fs_rows_.upload(rows, total); fs_ptr_.upload(ptr, total);
    fs_sums_.alloc(sums * std::min(8, nvb_), total);
    far_split_.n_blk = (int)row.size();
    far_split_.n_rows = (int)rows.size();
    far_split_.blk_row = fs_row_.p; far_split_.blk_begin = fs_begin_.p; far_split_.blk_end = fs_end_.p;
    far_split_.blk_part = fs_part_.p;
    far_split_.row = fs_rows_.p; far_split_.row_ptr = fs_ptr_.p;
    far_split_.part = fs_sums_.p;
    far_split_.part_vs = sums;
  }

  // ---- adjoint evaluation: the transpose of the evaluation's linear map, phase by phase in
  // reverse order with the transposed translations.  For the symmetric kernels (K(x, y) =
  // K(y, x)^T: laplace_poten, stokes_vel) every transposed point interaction is the same kernel
  // with sources and targets exchanged, and the V-list M2L of offset R transposes to the one of
  // offset -R (the check and equivalent lattices of a node coincide at radius RAD0).
  struct HostLists {  // forward lists kept on the host to build the transposed ones
    std::vector<int32_t> tleaf, u_ptr, u_items, far_ptr, far_node, x_node, x_ptr, x_items, s2m_node;
    std::vector<double> far_rad;
    std::vector<int32_t> v_partner, v_src_fc, v_trg_fc, offs, vsrc_depth, vtrg_depth;
    // the node table (real nodes, then the periodic images as (node, shift code))
    std::vector<double> center;
    std::vector<float> nsz;
    std::vector<int32_t> sb, se, tb, te;
    std::vector<std::pair<int32_t, int>> imgs;
  } h_;
  int64_t device_bytes_ = 0;  // of the plan itself

  struct AdjointPlan {
    const typename DeviceOps<Real>::Transposed* op = nullptr;  // the transposed operators
    // node table of the transposed lists: the forward one plus images of target-side nodes (a
    // forward item at shift s becomes, transposed, its target seen from the source at -s)
    DBuf<double> center;
    DBuf<float> nsz;
    DBuf<int32_t> sb, se, tb, te;
    const Real* bcT = nullptr;  // periodic boundary operator transposed (K1_ x K0_)
    DBuf<double> volpart;  // per-block partial sums of the volume-potential correction's transpose
    DBuf<Real> tden;     // adjoint input gathered into target order (k1 x n_trg per vector)
    DBuf<double> sval;   // adjoint output accumulated in source order (k0 x n_src per vector)
    DBuf<int32_t> iota;  // 0, 1, 2, ...: one item per row
    DBuf<int32_t> u_leaf, u_ptr, u_items;  // U list: source leaf <- target leaves
    int n_u = 0;
    DBuf<int32_t> w_node, w_ptr, w_items;  // W list: RAD0 surface of a source node <- target leaves
    int n_w = 0;
    DBuf<int32_t> x_leaf, x_ptr, x_node;   // X list: source leaf <- RAD0 check surfaces
    DBuf<int64_t> x_den;
    DBuf<double> x_rad;
    int n_x = 0;
    DBuf<int64_t> s2u_den;                 // S2U: source leaf <- its RAD1 check surface
    DBuf<double> s2u_rad;
    TileSet vt;                            // V list: source parents <- target parents
    DBuf<float> vrscale;                   // run scales of vt (fp16 Hadamard)
    DBuf<int32_t> v_fc;                    // first child of each transposed target slot
    DBuf<Real> fft_scal, ifft_scal;
    int n_vt = 0;
  };
  std::unique_ptr<AdjointPlan> adj_;

  // CSR of the transposed relation: for rows r with items it, the rows of item -> list of r
  // Groups (key, value, payload) triples by key (stable): the rows out_row (keys in increasing
  // order), their item ranges out_ptr and the values and payloads in forward order.
  static void group_by_key(const std::vector<int32_t>& keys, const std::vector<int32_t>& vals,
                           const std::vector<int32_t>& pay, int n_keys, std::vector<int32_t>& out_row,
                           std::vector<int32_t>& out_ptr, std::vector<int32_t>& out_items, std::vector<int32_t>& out_pay) {
    std::vector<int32_t> start(n_keys + 1, 0);
    for (int32_t k : keys) start[k + 1]++;
    for (int k = 0; k < n_keys; k++) start[k + 1] += start[k];
    std::vector<int32_t> flat(keys.size()), flatp(keys.size());
    std::vector<int32_t> fill = start;
    for (size_t i = 0; i < keys.size(); i++) {
      flat[fill[keys[i]]] = vals[i];
      flatp[fill[keys[i]]++] = pay[i];
    }
    out_row.clear(); out_ptr.assign(1, 0); out_items.clear(); out_pay.clear();
    for (int k = 0; k < n_keys; k++) {
      if (start[k + 1] == start[k]) continue;
      out_row.push_back(k);
      out_items.insert(out_items.end(), flat.begin() + start[k], flat.begin() + start[k + 1]);
      out_pay.insert(out_pay.end(), flatp.begin() + start[k], flatp.begin() + start[k + 1]);
      out_ptr.push_back((int32_t)out_items.size());
    }
  }

  void build_adjoint() {
    auto a = std::make_unique<AdjointPlan>();
    int64_t total = 0;
    const int N = n_nodes_;
    a->op = &ops_->transposed();
    a->tden.alloc((int64_t)k1_ * n_trg_ * nvb_, &total);
    a->sval.alloc((int64_t)k0_ * n_src_ * nvb_, &total);
    // the adjoint's node table and the transposition of a list with images: a forward item v of
    // row node r (v a source node, or an image (s, shift)) becomes item adj(r, -shift) of row s
    std::vector<double> ac = h_.center;
    std::vector<float> ansz = h_.nsz;
    std::vector<int32_t> asb = h_.sb, ase = h_.se, atb = h_.tb, ate = h_.te;
    std::unordered_map<int64_t, int32_t> aimg;
    auto real_of = [&](int32_t v, int& code) -> int32_t {
      if (v < N) { code = 13; return v; }
      code = h_.imgs[v - N].second;
      return h_.imgs[v - N].first;
    };
    auto adj = [&](int32_t node, int code) -> int32_t {
      if (code == 13) return node;
      const int neg = 26 - code;  // the negated shift
      const int64_t key = (int64_t)node * 27 + neg;
      auto it = aimg.find(key);
      if (it != aimg.end()) return it->second;
      const int32_t v = (int32_t)ansz.size();
      const int sh[3] = {neg % 3 - 1, (neg / 3) % 3 - 1, neg / 9 - 1};
      for (int d = 0; d < 3; d++) ac.push_back(h_.center[3 * (size_t)node + d] + sh[d]);
      ansz.push_back(h_.nsz[node]);
      asb.push_back(h_.sb[node]); ase.push_back(h_.se[node]);
      atb.push_back(h_.tb[node]); ate.push_back(h_.te[node]);
      aimg.emplace(key, v);
      return v;
    };
    auto transpose = [&](const std::vector<int32_t>& row_key, const std::vector<int32_t>& ptr,
                         const std::vector<int32_t>& items, std::vector<int32_t>& out_row, std::vector<int32_t>& out_ptr,
                         std::vector<int32_t>& out_items, std::vector<int32_t>& out_real) {
      std::vector<int32_t> keys(items.size()), vals(items.size()), real(items.size());
      for (size_t r = 0; r + 1 < ptr.size(); r++)
        for (int32_t i = ptr[r]; i < ptr[r + 1]; i++) {
          int code = 13;
          keys[i] = real_of(items[i], code);
          vals[i] = adj(row_key[r], code);
          real[i] = row_key[r];
        }
      group_by_key(keys, vals, real, N, out_row, out_ptr, out_items, out_real);
    };
    {
      std::vector<int32_t> iota(std::max<int>(n_tleaf_, n_s2m_) + 1);
      for (size_t i = 0; i < iota.size(); i++) iota[i] = (int32_t)i;
      a->iota.upload(iota, &total);
    }
    // U list
    {
      std::vector<int32_t> row, ptr, items, real;
      transpose(h_.tleaf, h_.u_ptr, h_.u_items, row, ptr, items, real);
      a->n_u = (int)row.size();
      a->u_leaf.upload(row, &total); a->u_ptr.upload(ptr, &total); a->u_items.upload(items, &total);
    }
    // W list: the far items after each target leaf's own L2T surface
    {
      std::vector<int32_t> key, ptr{0}, items;
      for (size_t r = 0; r < h_.tleaf.size(); r++) {
        for (int32_t i = h_.far_ptr[r]; i < h_.far_ptr[r + 1]; i++)
          if (h_.far_rad[i] == kRad0) items.push_back(h_.far_node[i]);
        key.push_back(h_.tleaf[r]);
        ptr.push_back((int32_t)items.size());
      }
      std::vector<int32_t> row, tptr, titems, treal;
      transpose(key, ptr, items, row, tptr, titems, treal);
      a->n_w = (int)row.size();
      a->w_node.upload(row, &total); a->w_ptr.upload(tptr, &total); a->w_items.upload(titems, &total);
    }
    // X list
    {
      std::vector<int32_t> row, ptr, items, real;
      transpose(h_.x_node, h_.x_ptr, h_.x_items, row, ptr, items, real);
      a->n_x = (int)row.size();
      std::vector<int64_t> den(items.size());  // the check potentials of the real nodes
      for (size_t i = 0; i < items.size(); i++) den[i] = (int64_t)real[i] * K1_;
      a->x_leaf.upload(row, &total); a->x_ptr.upload(ptr, &total); a->x_node.upload(items, &total);
      a->x_den.upload(den, &total);
      a->x_rad.upload(std::vector<double>(items.size(), kRad0), &total);
    }
    // S2U: row r reads its own check potential, chk row r
    {
      std::vector<int64_t> den(n_s2m_);
      for (int r = 0; r < n_s2m_; r++) den[r] = (int64_t)r * K1_;
      a->s2u_den.upload(den, &total);
      a->s2u_rad.upload(std::vector<double>(n_s2m_, kRad1), &total);
    }
    // V list: new targets are the source parents, new sources the target parents; the pair
    // (t, R, s) of the evaluation becomes (s, -R, t), whose offset index is that of 26 - R
    {
      const int n_off = n_off_;
      std::vector<int> neg(n_off, -1);
      for (int o = 0; o < n_off; o++)
        for (int o2 = 0; o2 < n_off; o2++)
          if (h_.offs[o2] == 26 - h_.offs[o]) neg[o] = o2;
      for (int o = 0; o < n_off; o++)
        if (neg[o] < 0) throw Error(kErrInternal, "V-list offsets are not closed under negation");
      std::vector<int32_t> full((size_t)n_vsrc_ * n_off, -1);
      std::vector<char> has(n_vsrc_, 0);
      for (int t = 0; t < n_vtrg_; t++)
        for (int o = 0; o < n_off; o++) {
          const int32_t sl = h_.v_partner[(size_t)t * n_off + o];
          if (sl < 0) continue;
          full[(size_t)sl * n_off + neg[o]] = t;
          has[sl] = 1;
        }
      std::vector<int32_t> partner, fc;
      std::vector<Real> fscal(n_vtrg_), iscal;
      const KernelInfo& ki = O_.ker;
      for (int sl = 0; sl < n_vsrc_; sl++) {
        if (!has[sl]) continue;
        partner.insert(partner.end(), full.begin() + (size_t)sl * n_off, full.begin() + (size_t)(sl + 1) * n_off);
        fc.push_back(h_.v_src_fc[sl]);
        iscal.push_back((Real)std::pow(2.0, ki.trg_scal * (h_.vsrc_depth[sl] + 1)));
      }
      for (int t = 0; t < n_vtrg_; t++) fscal[t] = (Real)std::pow(2.0, ki.src_scal * (h_.vtrg_depth[t] + 1));
      a->n_vt = (int)fc.size();
      build_tiles(partner, a->n_vt, n_vtrg_, a->vt, &total);
      if (split_) a->vrscale.alloc((int64_t)2 * std::max(1, a->vt.n) * vlist_nv_, &total);
      a->v_fc.upload(fc, &total);
      a->fft_scal.upload(fscal, &total);
      a->ifft_scal.upload(iscal, &total);
    }
    a->center.upload(ac, &total);
    a->nsz.upload(ansz, &total);
    a->sb.upload(asb, &total); a->se.upload(ase, &total);
    a->tb.upload(atb, &total); a->te.upload(ate, &total);
    if (bndry_ != kFreeSpace) {
      a->bcT = ops_->bc(bndry_, true);
      if (vol_) a->volpart.alloc((int64_t)K::vol_adjoint_blocks() * 3 * nvb_, &total);
    }
    device_bytes_ += total;
    adj_ = std::move(a);
  }

  void adjoint_one(const double* d_g, double* d_out, double den_scale, double out_scale, int nv) {
    AdjointPlan& a = *adj_;
    const int ek = O_.ker.exp_kind;  // == the point kernel for the symmetric kernels
    const int64_t g_vs = (int64_t)k1_ * n_trg_, o_vs = (int64_t)k0_ * n_src_;
    const int sp = tuning.gemm_split_blocks;
    // scatter^T: the adjoint input in sorted target order (times the output scale)
    K::gather_density(st_, n_trg_, k1_, d_g, trg_perm_.p, out_scale, a.tden.p, nv, g_vs);
    K::fill(st_, eq_.p, eq_vs_ * nv);
    K::fill(st_, dn_.p, dn_vs_ * nv);
    K::fill64(st_, a.sval.p, o_vs * nv);
    // (volume-potential correction)^T: the targets' weighted sums onto the root's equivalent density
    if (vol_)
      K::vol_correction_adjoint(st_, O_.ker.pt_kind, n_trg_, txa_.p, a.tden.p, K0_, e0_, eq_.p, a.volpart.p, nv, g_vs, eq_vs_);
    // U list^T: target points -> source points of the leaves listing them
    K::p2p_points(st_, ek, a.n_u, a.u_leaf.p, a.u_ptr.p, a.u_items.p, a.sb.p, a.se.p, a.tb.p, a.te.p,
                  a.center.p, sx64_.p, n_src_, tx64_.p, a.tden.p, n_trg_, a.sval.p, true, nv, g_vs, o_vs);
    // (L2T P2P)^T: target points -> their leaf's downward equivalent surface (RAD1)
    K::p2p_surface(st_, ek, n_tleaf_, t_leaf_.p, a.iota.p, t_leaf_.p, a.tb.p, a.te.p, a.center.p, a.nsz.p, kRad1,
                   ops_->unit_surf.p, ns_, tx_.p, a.tden.p, n_trg_, eq_.p, l2t_rc_.p, K0_, true, nv, g_vs, eq_vs_);
    // (W list M2T)^T: target points -> upward equivalent surfaces (RAD0) of their W sources
    K::p2p_surface(st_, ek, a.n_w, a.w_node.p, a.w_ptr.p, a.w_items.p, a.tb.p, a.te.p, a.center.p, a.nsz.p, kRad0,
                   ops_->unit_surf.p, ns_, tx_.p, a.tden.p, n_trg_, eq_.p, a.w_node.p, K0_, true, nv, g_vs, eq_vs_);
    // D2T GEMMs^T: equivalent -> check potential of each target leaf
    pair(a.op->d2t_pair, a.op->dc2de1, a.op->dc2de0, n_l2t_, K0_, rd_, K1_, eq_.p, l2t_rc_.p, nullptr, l2t_seq_.p, dn_.p, l2t_ra_.p,
         l2t_alpha_.p, true, nv, eq_vs_, dn_vs_);
    // D2D^T, bottom-up: parent += [8 children] x [D2D_0 .. D2D_7]^T
    for (int l = max_depth_; l >= dn_min_ + 1; l--) {
      const LevelRows& L = *l2l_[l - 1];
      if (ops_->d2d_fact && L.n >= kFactorRows) {
        K::gemm_rows(st_, L.n, rd_, 8 * K1_, dn_.p, L.rc.p, K1_, a.op->d2dr.p, ctmp_.p, lvl_seq_.p, rd_, nullptr, false,
                     gemm_work_.p, gemm_work_elems_, sp, nv, dn_vs_, ctmp_vs_);
        K::gemm_rows(st_, L.n, K1_, rd_, ctmp_.p, lvl_seq_.p, rd_, a.op->dc2de0.p, dn_.p, L.ra.p, K1_, nullptr, true,
                     gemm_work_.p, gemm_work_elems_, sp, nv, ctmp_vs_, dn_vs_);
      } else {
        K::gemm_rows(st_, L.n, K1_, 8 * K1_, dn_.p, L.rc.p, K1_, a.op->d2d.p, dn_.p, L.ra.p, K1_, nullptr, true, gemm_work_.p,
                     gemm_work_elems_, sp, nv, dn_vs_, dn_vs_);
      }
    }
    // (periodic boundary)^T: root equivalent density += root check potential x BC^T
    if (bndry_ != kFreeSpace)
      K::gemm_rows(st_, 1, K0_, K1_, dn_.p, lvl_seq_.p, K1_, a.bcT, eq_.p, lvl_seq_.p, K0_, nullptr, true, gemm_work_.p,
                   gemm_work_elems_, sp, nv, dn_vs_, eq_vs_);
    // V list^T: the M2L of offset -R from the target parents' children to the source parents'
    // (the spectra buffers swap roles: Y_ holds the new sources, X_ the new targets)
    for (int v = 0; v < nv; v += vlist_nv_) {
      const int g = std::min(vlist_nv_, nv - v);
      K::fft_up(st_, n_vtrg_, v_trg_fc_.p, dn_.p + v * dn_vs_, K1_, e1_, m_, ops_->lattice.p, ops_->lattice_inv.p, a.fft_scal.p,
                Y_.p, split_ ? vbound_.p : nullptr, g, dn_vs_, y_vs_, bound_vs_);
      K::hadamard_tiled(st_, a.vt.n, M_dim_, e0_, e1_, n_off_, a.vt.t0.p, a.vt.u0.p, a.vt.usrc.p, a.vt.d0.p, a.vt.dent.p,
                        a.vt.uidx.p, a.vt.gmask.p, v_offsets_.p, ops_->V.p, Y_.p, X_.p, tuning.hadamard_tpb,
                        split_ ? &hparts(a.vrscale) : nullptr, g, y_vs_, x_vs_);
      K::ifft_down(st_, a.n_vt, a.v_fc.p, X_.p, eq_.p + v * eq_vs_, K0_, e0_, m_, ops_->lattice.p, ops_->lattice_inv.p, ns_,
                   a.ifft_scal.p, g, x_vs_, eq_vs_);
    }
    // (X list S2L)^T: downward check surfaces (RAD0) -> source points
    K::far_points(st_, ek, a.n_x, a.x_leaf.p, a.x_ptr.p, a.x_node.p, a.x_den.p, a.x_rad.p, a.sb.p, a.se.p,
                  a.center.p, a.nsz.p, ops_->unit_surf.p, ns_, sx_.p, n_src_, dn_.p, a.sval.p, true, nv, dn_vs_, o_vs);
    // U2U^T, top-down: [8 children] += parent x [U2U_0 .. U2U_7]^T
    for (int l = up_min_; l <= max_depth_ - 1; l++) {
      const LevelRows& L = *m2m_[l];
      if (ops_->u2u_fact && L.n >= kFactorRows) {
        K::gemm_rows(st_, L.n, ru_, K0_, eq_.p, L.rc.p, K0_, a.op->uc2ue1.p, ctmp_.p, lvl_seq_.p, ru_, nullptr, false,
                     gemm_work_.p, gemm_work_elems_, sp, nv, eq_vs_, ctmp_vs_);
        K::gemm_rows(st_, L.n, 8 * K0_, ru_, ctmp_.p, lvl_seq_.p, ru_, a.op->u2ur.p, eq_.p, L.ra.p, K0_, nullptr, true,
                     gemm_work_.p, gemm_work_elems_, sp, nv, ctmp_vs_, eq_vs_);
      } else {
        K::gemm_rows(st_, L.n, 8 * K0_, K0_, eq_.p, L.rc.p, K0_, a.op->u2u.p, eq_.p, L.ra.p, K0_, nullptr, true, gemm_work_.p,
                     gemm_work_elems_, sp, nv, eq_vs_, eq_vs_);
      }
    }
    // S2U GEMMs^T: upward equivalent -> check potential of each source leaf
    pair(a.op->s2u_pair, a.op->uc2ue1, a.op->uc2ue0, n_s2m_, K0_, ru_, K1_, eq_.p, s2m_node_.p, nullptr, s2m_orow_.p, chk_.p,
         s2m_orow_.p, s2m_alpha_.p, false, nv, eq_vs_, chk_vs_);
    // (S2U P2P)^T: upward check surface (RAD1) -> the leaf's source points
    K::far_points(st_, ek, n_s2m_, s2m_node_.p, a.iota.p, s2m_node_.p, a.s2u_den.p, a.s2u_rad.p, a.sb.p, a.se.p,
                  a.center.p, a.nsz.p, ops_->unit_surf.p, ns_, sx_.p, n_src_, chk_.p, a.sval.p, true, nv, chk_vs_, o_vs);
    // gather^T: back to the input order of the sources (times the density scale)
    K::scatter_output(st_, n_src_, k0_, a.sval.p, src_perm_.p, den_scale, d_out, nv, o_vs);
  }

 public:
  bool adjoint_supported() const override { return O_.ker.pt_kind == O_.ker.exp_kind; }
  void evaluate_adjoint(const double* d_g, double* d_out, int n_vec, double den_scale, double out_scale) override {
    if (!adjoint_supported())
      throw Error(kErrUnsupported, std::string("the adjoint evaluation needs a symmetric kernel (laplace_poten, stokes_vel); ") +
                                       O_.ker.name + " is not");
    if (n_vec < 1) throw Error(kErrInvalidArgument, "n_vec must be >= 1");
    if (!adj_) build_adjoint();
    for (int v = 0; v < n_vec; v += nvb_)
      adjoint_one(d_g + (int64_t)v * k1_ * n_trg_, d_out + (int64_t)v * k0_ * n_src_, den_scale, out_scale,
                  std::min(nvb_, n_vec - v));
  }

 private:
  void evaluate_one(const double* d_den, double* d_out, double den_scale, double out_scale, int nv,
                    const double* const* den_slot = nullptr, double* const* out_slot = nullptr) {
    const int pk = O_.ker.pt_kind, ek = O_.ker.exp_kind;
    const int64_t den_vs = (int64_t)k0_ * n_src_, val_vs = (int64_t)k1_ * n_trg_;
    const int sp = tuning.gemm_split_blocks;
    mark(0);
    K::begin(st_, n_src_, k0_, d_den, src_perm_.p, den_scale, sden_.p, nv, den_vs, eq_.p, eq_vs_ * nv, dn_.p, dn_vs_ * nv,
             den_slot);
    mark(1);
    // S2U: sources -> upward check surface (RAD1), then check -> equivalent
    K::p2p_surface(st_, ek, n_s2m_, s2m_node_.p, s2m_ptr_.p, s2m_items_.p, src_begin_.p, src_end_.p, center_.p, node_size_.p,
                   kRad1, ops_->unit_surf.p, ns_, sx_.p, sden_.p, n_src_, chk_.p, s2m_orow_.p, K1_, false, nv, den_vs, chk_vs_);
    mark(2);
    pair(ops_->s2u_pair, ops_->uc2ue0, ops_->uc2ue1, n_s2m_, K1_, ru_, K0_, chk_.p, s2m_orow_.p, s2m_alpha_.p, s2m_orow_.p, eq_.p,
         s2m_node_.p, nullptr, false, nv, chk_vs_, eq_vs_);
    mark(3);
    // U2U, bottom-up: parent row = [8 children] x stacked U2U
    for (int l = max_depth_ - 1; l >= up_min_; l--) {
      const LevelRows& L = *m2m_[l];
      if (ops_->u2u_fact && L.n >= kFactorRows) {  // [8 children] -> rank coordinates -> parent
        K::gemm_rows(st_, L.n, ru_, 8 * K0_, eq_.p, L.ra.p, K0_, ops_->u2ur.p, ctmp_.p, lvl_seq_.p, ru_, nullptr, false,
                     gemm_work_.p, gemm_work_elems_, sp, nv, eq_vs_, ctmp_vs_);
        K::gemm_rows(st_, L.n, K0_, ru_, ctmp_.p, lvl_seq_.p, ru_, ops_->uc2ue1.p, eq_.p, L.rc.p, K0_, nullptr, false,
                     gemm_work_.p, gemm_work_elems_, sp, nv, ctmp_vs_, eq_vs_);
      } else {
        K::gemm_rows(st_, L.n, K0_, 8 * K0_, eq_.p, L.ra.p, K0_, ops_->u2u.p, eq_.p, L.rc.p, K0_, nullptr, false, gemm_work_.p,
                     gemm_work_elems_, sp, nv, eq_vs_, eq_vs_);
      }
    }
    // periodic images beyond the root's colleagues: root check potential += root equivalent x BC
    if (bndry_ != kFreeSpace)
      K::gemm_rows(st_, 1, K1_, K0_, eq_.p, lvl_seq_.p, K0_, bc_, dn_.p, lvl_seq_.p, K1_, nullptr, true, gemm_work_.p,
                   gemm_work_elems_, sp, nv, eq_vs_, dn_vs_);
    mark(4);
    // X list: source points -> downward check surface (RAD0)
    K::p2p_surface(st_, ek, n_x_, x_node_.p, x_ptr_.p, x_items_.p, src_begin_.p, src_end_.p, center_.p, node_size_.p, kRad0,
                   ops_->unit_surf.p, ns_, sx_.p, sden_.p, n_src_, dn_.p, x_orow_.p, K1_, true, nv, den_vs, dn_vs_);
    mark(5);
    // V list: passes of up to vlist_nv_ vectors through the spectra buffers (with several passes
    // the three sub-phases are timed per pass and summed)
    const int n_pass = (nv + vlist_nv_ - 1) / vlist_nv_;
    const bool sub = timing_ && n_pass > 1;
    if (sub) ensure_vlist_events(n_pass);
    for (int p = 0; p < n_pass; p++) {
      const int v = p * vlist_nv_, g = std::min(vlist_nv_, nv - v);
      if (sub) HIP_CHECK(hipEventRecord(vev_[4 * p], st_));
      K::fft_up(st_, n_vsrc_, v_src_fc_.p, eq_.p + v * eq_vs_, K0_, e0_, m_, ops_->lattice.p, ops_->lattice_inv.p, v_src_scal_.p,
                X_.p, split_ ? vbound_.p : nullptr, g, eq_vs_, x_vs_, bound_vs_);
      if (sub) HIP_CHECK(hipEventRecord(vev_[4 * p + 1], st_));
      if (n_pass == 1) mark(6);
      K::hadamard_tiled(st_, vt_.n, M_dim_, e0_, e1_, n_off_, vt_.t0.p, vt_.u0.p, vt_.usrc.p, vt_.d0.p, vt_.dent.p,
                        vt_.uidx.p, vt_.gmask.p, v_offsets_.p, ops_->V.p, X_.p, Y_.p, tuning.hadamard_tpb,
                        split_ ? &hparts(vrscale_) : nullptr, g, x_vs_, y_vs_);
      if (sub) HIP_CHECK(hipEventRecord(vev_[4 * p + 2], st_));
      if (n_pass == 1) mark(7);
      K::ifft_down(st_, n_vtrg_, v_trg_fc_.p, Y_.p, dn_.p + v * dn_vs_, K1_, e1_, m_, ops_->lattice.p, ops_->lattice_inv.p, ns_,
                   v_trg_scal_.p, g, y_vs_, dn_vs_);
      if (sub) HIP_CHECK(hipEventRecord(vev_[4 * p + 3], st_));
    }
    if (n_pass > 1) {
      mark(6);
      mark(7);
    }
    mark(8);
    // D2D, top-down: 8 children rows += parent x [D2D_0 .. D2D_7]
    for (int l = dn_min_ + 1; l <= max_depth_; l++) {
      const LevelRows& L = *l2l_[l - 1];
      if (ops_->d2d_fact && L.n >= kFactorRows) {  // parent check -> rank coordinates -> [8 children]
        K::gemm_rows(st_, L.n, rd_, K1_, dn_.p, L.ra.p, K1_, ops_->dc2de0.p, ctmp_.p, lvl_seq_.p, rd_, nullptr, false,
                     gemm_work_.p, gemm_work_elems_, sp, nv, dn_vs_, ctmp_vs_);
        K::gemm_rows(st_, L.n, 8 * K1_, rd_, ctmp_.p, lvl_seq_.p, rd_, ops_->d2dr.p, dn_.p, L.rc.p, K1_, nullptr, true,
                     gemm_work_.p, gemm_work_elems_, sp, nv, ctmp_vs_, dn_vs_);
      } else {
        K::gemm_rows(st_, L.n, 8 * K1_, K1_, dn_.p, L.ra.p, K1_, ops_->d2d.p, dn_.p, L.rc.p, K1_, nullptr, true, gemm_work_.p,
                     gemm_work_elems_, sp, nv, dn_vs_, dn_vs_);
      }
    }
    mark(9);
    // D2T: check -> equivalent
    pair(ops_->d2t_pair, ops_->dc2de0, ops_->dc2de1, n_l2t_, K1_, rd_, K0_, dn_.p, l2t_ra_.p, l2t_alpha_.p, l2t_seq_.p, eq_.p,
         l2t_rc_.p, nullptr, false, nv, dn_vs_, eq_vs_);
    mark(10);
    // equivalent surfaces -> targets (own downward equivalent + W list)
    K::far_points(st_, pk, n_tleaf_, t_leaf_.p, far_ptr_.p, far_node_.p, far_den_.p, far_rad_.p, trg_begin_.p, trg_end_.p,
                  center_.p, node_size_.p, ops_->unit_surf.p, ns_, tx_.p, n_trg_, eq_.p, tval_.p, false, nv, eq_vs_, val_vs,
                  far_split_);
    mark(11);
    // U list: near-field P2P
    K::p2p_points(st_, pk, n_tleaf_, t_leaf_.p, u_ptr_.p, u_items_.p, trg_begin_.p, trg_end_.p, src_begin_.p, src_end_.p,
                  center_.p, tx64_.p, n_trg_, sx64_.p, sden_.p, n_src_, tval_.p, true, nv, den_vs, val_vs);
    if (vol_)  // minus the root's total equivalent density times the analytic volume potential
      K::vol_correction(st_, pk, n_trg_, txa_.p, eq_.p, K0_, e0_, tval_.p, nv, eq_vs_, val_vs);
    mark(12);
    // targets not in any leaf with targets are impossible; every target lies in exactly one leaf
    K::scatter_output(st_, n_trg_, k1_, tval_.p, trg_perm_.p, out_scale, d_out, nv, val_vs, out_slot);
    mark(13);
    if (timing_) {
      HIP_CHECK(hipEventSynchronize(ev_[kPhaseCount]));
      for (int p = 0; p < kPhaseCount; p++) {
        float ms = 0;
        HIP_CHECK(hipEventElapsedTime(&ms, ev_[p], ev_[p + 1]));
        phase_ms[p] = ms;
      }
      if (n_pass > 1) {
        phase_ms[kPhFFT] = phase_ms[kPhHadamard] = phase_ms[kPhIFFT] = 0;
        for (int v = 0; v < n_pass; v++)
          for (int q = 0; q < 3; q++) {
            float ms = 0;
            HIP_CHECK(hipEventElapsedTime(&ms, vev_[4 * v + q], vev_[4 * v + q + 1]));
            phase_ms[kPhFFT + q] += ms;
          }
      }
    }
  }
};

}  // namespace

std::unique_ptr<DevicePlanBase> make_plan(const Octree& T, const Operators& O, const double* src_xyz, const double* trg_xyz,
                                          int precision, int n_vec_max, hipStream_t stream,
                                          std::shared_ptr<DeviceOpsBase> ops) {
  if (precision == 0)
    return std::make_unique<DevicePlan<double>>(T, O, std::static_pointer_cast<DeviceOps<double>>(ops), src_xyz, trg_xyz,
                                                n_vec_max, stream);
  if (precision == 1)
    return std::make_unique<DevicePlan<float>>(T, O, std::static_pointer_cast<DeviceOps<float>>(ops), src_xyz, trg_xyz,
                                               n_vec_max, stream);
  throw Error(kErrInvalidArgument, "precision must be 0 (fp64) or 1 (mixed fp32)");
}

std::shared_ptr<DeviceOpsBase> make_device_ops(const Operators& O, int precision) {
  if (precision == 0) return std::make_shared<DeviceOps<double>>(O);
  if (precision == 1) return std::make_shared<DeviceOps<float>>(O);
  throw Error(kErrInvalidArgument, "precision must be 0 (fp64) or 1 (mixed fp32)");
}

}  // namespace pvfmm_amd
