// An operator set on the device: the translations and V-list transfer blocks in the working
// precision, shared by every tree plan of one operator handle on one device.  Made on the first
// setup and kept by the handle (a plan holds a reference), so a tree set up again pays for its
// own lists only.
#pragma once
#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <type_traits>
#include <vector>

#include <hip/hip_runtime_api.h>

#include "device_fmm.hpp"
#include "kernels.hpp"
#include "operators.hpp"
#include "transfer.hpp"

namespace pvfmm_amd {

template <typename T>
struct DBuf {
  T* p = nullptr;
  int64_t n = 0;
  DBuf() = default;
  DBuf(const DBuf&) = delete;
  DBuf& operator=(const DBuf&) = delete;
  ~DBuf() { if (p) (void)hipFree(p); }
  void alloc(int64_t count, int64_t* total) {
    if (p) { (void)hipFree(p); p = nullptr; }
    n = count;
    if (count > 0) {
      HIP_CHECK(hipMalloc(&p, sizeof(T) * count));
      if (total) *total += sizeof(T) * count;
    }
  }
  void upload(const std::vector<T>& v, int64_t* total) {
    alloc((int64_t)v.size(), total);
    if (!v.empty()) HIP_CHECK(hipMemcpy(p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice));
  }
};

template <typename Real>
class DeviceOps final : public DeviceOpsBase {
 public:
  // check -> equivalent factors with the rank padded to a multiple of 16 (zero columns of the
  // first factor, zero rows of the second), so the GEMM operands stay 4-vector aligned
  int ru = 0, rd = 0;
  DBuf<Real> uc2ue0, uc2ue1, dc2de0, dc2de1, u2u, d2d;
  // U2U and D2D through the rank of the check-to-equivalent factors, when 9 r < 8 K.  The
  // composite translations are u2u = T uc2ue1 (T: 8 K0 x r, uc2ue1: r x K0 with orthonormal rows)
  // and d2d = dc2de0 B (dc2de0: K1 x r with orthogonal columns of norms 1/s_j, B: r x 8 K1), so
  // T = u2u uc2ue1^T and B = diag(s^2) dc2de0^T d2d (include/fmm_pts.txx:582-643 forms the same
  // products).  Applied as two GEMMs they cost 9 K r instead of 8 K^2 multiply-adds per row.
  bool u2u_fact = false, d2d_fact = false;
  DBuf<Real> u2ur, d2dr;  // 8 K0 x ru, rd x 8 K1
  // the factors packed for the one-launch product of the leaves' maps, where their shapes fit it and
  // some number of rows takes it
  struct PackedPair {
    DBuf<Real> B1, B2;
    bool use = false;
  };
  PackedPair s2u_pair, d2t_pair;  // uc2ue0 uc2ue1, dc2de0 dc2de1
  DBuf<Real> unit_surf;
  DBuf<int32_t> lattice, lattice_inv;
  VGrid grid;
  DBuf<Real> V;          // transfer blocks in real form (FP64)
  DBuf<uint16_t> Vh;     // as two fp16 parts (FP32), with 1 / tau_f
  DBuf<float> vtinv;
  bool split = false;    // FP32: the fp16 Hadamard kernels

  explicit DeviceOps(const Operators& O) : O_(O) {
    int64_t sum = 0, *total = &sum;
    const int K0 = O.K0(), K1 = O.K1(), e0 = O.ker.e0, e1 = O.ker.e1;
    Stream st;
    const hipStream_t s = st.s;
    ru = (O.rank_u + 15) / 16 * 16;
    rd = (O.rank_d + 15) / 16 * 16;
    DBuf<double> a, b, c, d;
    auto padded = [&](DBuf<double>& in, const std::vector<double>& v, int r0, int c0, DBuf<Real>& out, int rows, int cols) {
      in.upload(v, nullptr);
      out.alloc((int64_t)rows * cols, total);
      convert_matrix<Real>(s, in.p, r0, c0, out.p, rows, cols);
    };
    padded(a, O.uc2ue0, K1, O.rank_u, uc2ue0, K1, ru);
    padded(b, O.uc2ue1, O.rank_u, K0, uc2ue1, ru, K0);
    padded(c, O.dc2de0, K1, O.rank_d, dc2de0, K1, rd);
    padded(d, O.dc2de1, O.rank_d, K0, dc2de1, rd, K0);
    DBuf<double> u, t;
    padded(u, O.u2u, 8 * K0, K0, u2u, 8 * K0, K0);
    padded(t, O.d2d, K1, 8 * K1, d2d, K1, 8 * K1);
    u2u_fact = 9 * ru < 8 * K0;
    d2d_fact = 9 * rd < 8 * K1;
    if (u2u_fact || d2d_fact) {
      std::vector<int32_t> iota(std::max(8 * K0, std::max(K1, std::max(ru, rd))));
      for (size_t i = 0; i < iota.size(); i++) iota[i] = (int32_t)i;
      DBuf<int32_t> di;
      di.upload(iota, nullptr);
      DBuf<double> tr, prod;
      if (u2u_fact) {
        tr.alloc((int64_t)K0 * O.rank_u, nullptr);
        prod.alloc((int64_t)8 * K0 * O.rank_u, nullptr);
        convert_matrix<double>(s, b.p, O.rank_u, K0, tr.p, K0, O.rank_u, true);
        DeviceKernels<double>::gemm_rows(s, 8 * K0, O.rank_u, K0, u.p, di.p, K0, tr.p, prod.p, di.p, O.rank_u, nullptr, false);
        u2ur.alloc((int64_t)8 * K0 * ru, total);
        convert_matrix<Real>(s, prod.p, 8 * K0, O.rank_u, u2ur.p, 8 * K0, ru);
        HIP_CHECK(hipStreamSynchronize(s));  // tr and prod are used again
      }
      if (d2d_fact) {
        std::vector<double> inv2(O.rank_d, 0.0);
        for (int i = 0; i < K1; i++)
          for (int j = 0; j < O.rank_d; j++) inv2[j] += O.dc2de0[(size_t)i * O.rank_d + j] * O.dc2de0[(size_t)i * O.rank_d + j];
        for (double& v : inv2) v = 1.0 / v;
        DBuf<double> al;
        al.upload(inv2, nullptr);
        tr.alloc((int64_t)O.rank_d * K1, nullptr);
        prod.alloc((int64_t)O.rank_d * 8 * K1, nullptr);
        convert_matrix<double>(s, c.p, K1, O.rank_d, tr.p, O.rank_d, K1, true);
        DeviceKernels<double>::gemm_rows(s, O.rank_d, 8 * K1, K1, tr.p, di.p, K1, t.p, prod.p, di.p, 8 * K1, al.p, false);
        d2dr.alloc((int64_t)rd * 8 * K1, total);
        convert_matrix<Real>(s, prod.p, O.rank_d, 8 * K1, d2dr.p, rd, 8 * K1);
        HIP_CHECK(hipStreamSynchronize(s));
      }
    }
    HIP_CHECK(hipStreamSynchronize(s));
    DeviceKernels<Real>::gemm_pair_init();
    pack_pair(s, uc2ue0, K1, ru, uc2ue1, K0, s2u_pair, total);
    pack_pair(s, dc2de0, K1, rd, dc2de1, K0, d2t_pair, total);
    HIP_CHECK(hipStreamSynchronize(s));
    unit_surf.upload(std::vector<Real>(O.unit_surf.begin(), O.unit_surf.end()), total);
    lattice.upload(O.lattice, total);
    std::vector<int32_t> inv((size_t)O.m * O.m * O.m, -1);
    for (int p = 0; p < O.ns; p++)
      inv[((size_t)O.lattice[3 * p + 2] * O.m + O.lattice[3 * p + 1]) * O.m + O.lattice[3 * p]] = p;
    lattice_inv.upload(inv, total);
    grid = v_grid(O.m);
    DBuf<double> G;
    spectra(s, G);
    if constexpr (std::is_same<Real, float>::value) {
      Vh.alloc((int64_t)13 * grid.M * e0 * e1 * 2 * 512, total);
      vtinv.alloc(grid.M, total);
      transfer_fp16(s, e0, e1, grid.M, G.p, Vh.p, vtinv.p);
      split = true;
    } else {
      V.alloc((int64_t)27 * grid.M * e0 * e1 * 256, total);
      transfer_real(s, e0, e1, grid.M, G.p, V.p);
    }
    HIP_CHECK(hipStreamSynchronize(s));
    bytes_ = sum;
  }

  int64_t bytes() const override { return bytes_; }  // grows with the first bc() and transposed()

  // Boundary operator of a periodic boundary type (K0 x K1), and transposed
  const Real* bc(int bndry, bool transposed) {
    std::lock_guard<std::mutex> lock(mutex_);
    DBuf<Real>& B = bc_[transposed][bndry];
    if (!B.p) {
      const std::vector<double>& h = O_.bc[bndry];
      if (h.size() != (size_t)O_.K0() * O_.K1()) throw Error(kErrInternal, "periodic tree without its boundary operator");
      transpose_or_copy(h, O_.K0(), O_.K1(), B, transposed);
    }
    return B.p;
  }
  // The transposed operators of the adjoint evaluation, in the padded layouts of the forward ones
  struct Transposed {
    DBuf<Real> uc2ue0, uc2ue1, dc2de0, dc2de1, u2u, d2d, u2ur, d2dr;
    PackedPair d2t_pair, s2u_pair;  // dc2de1^T dc2de0^T, uc2ue1^T uc2ue0^T
  };
  const Transposed& transposed() {
    std::lock_guard<std::mutex> lock(mutex_);
    if (!tr_) {
      auto t = std::make_unique<Transposed>();
      const int K0 = O_.K0(), K1 = O_.K1();
      int64_t sum = 0;
      Stream st;
      auto turn = [&](const DBuf<Real>& in, int rows, int cols, DBuf<Real>& out) {
        if (!in.p) return;
        out.alloc((int64_t)rows * cols, &sum);
        transpose_matrix<Real>(st.s, in.p, rows, cols, out.p);
      };
      turn(uc2ue0, K1, ru, t->uc2ue0);
      turn(uc2ue1, ru, K0, t->uc2ue1);
      turn(dc2de0, K1, rd, t->dc2de0);
      turn(dc2de1, rd, K0, t->dc2de1);
      turn(u2u, 8 * K0, K0, t->u2u);
      turn(d2d, K1, 8 * K1, t->d2d);
      turn(u2ur, 8 * K0, ru, t->u2ur);
      turn(d2dr, rd, 8 * K1, t->d2dr);
      pack_pair(st.s, t->dc2de1, K0, rd, t->dc2de0, K1, t->d2t_pair, &sum);
      pack_pair(st.s, t->uc2ue1, K0, ru, t->uc2ue0, K1, t->s2u_pair, &sum);
      HIP_CHECK(hipStreamSynchronize(st.s));
      bytes_ += sum;
      tr_ = std::move(t);
    }
    return *tr_;
  }

 private:
  struct Stream {
    hipStream_t s = nullptr;
    Stream() { HIP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking)); }
    ~Stream() { (void)hipStreamDestroy(s); }
  };
  void pack_pair(hipStream_t s, const DBuf<Real>& f0, int K, int r, const DBuf<Real>& f1, int N, PackedPair& p, int64_t* total) {
    using D = DeviceKernels<Real>;
    p.use = D::gemm_pair_fits(K, r) && D::gemm_pair_pays(K, 4 * (int64_t)K);
    if (!p.use) return;
    p.B1.alloc(D::packed_size(K, r), total);
    p.B2.alloc(D::packed_size(r, N), total);
    D::pack_matrix(s, f0.p, K, r, p.B1.p);
    D::pack_matrix(s, f1.p, r, N, p.B2.p);
  }
  void spectra(hipStream_t s, DBuf<double>& G) {
    G.alloc((int64_t)2 * 343 * O_.ker.e0 * O_.ker.e1 * grid.M, nullptr);
    transfer_spectra(s, O_.ker.exp_kind, O_.m, G.p);
  }
  void transpose_or_copy(const std::vector<double>& h, int rows, int cols, DBuf<Real>& out, bool transposed) {
    Stream st;
    DBuf<double> in;
    in.upload(h, nullptr);
    int64_t sum = 0;
    out.alloc((int64_t)rows * cols, &sum);
    convert_matrix<Real>(st.s, in.p, rows, cols, out.p, transposed ? cols : rows, transposed ? rows : cols, transposed);
    HIP_CHECK(hipStreamSynchronize(st.s));
    bytes_ += sum;
  }

  const Operators& O_;
  std::atomic<int64_t> bytes_{0};  // read by plans that other threads set up
  std::mutex mutex_;
  DBuf<Real> bc_[2][4];
  std::unique_ptr<Transposed> tr_;
};

}  // namespace pvfmm_amd
