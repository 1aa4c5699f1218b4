// Internal interface between the SGS-closure C ABI (sgs_api.hip) and its
// kernels (sgs_kernels.hip).  Not installed.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "psdns_internal.h"

struct psdns_ctx;

namespace psdns {

// Access to a step context for the library's other C-ABI files: the context
// made ready (a deferred update run; with clobber, the next stage update
// refused because the work arrays will be overwritten), its launch context
// (the physical array allocated when need_ux), and its synchronisation.
int ctx_access(psdns_ctx* c, bool clobber, bool need_ux, Ctx* out, int* n);
int ctx_sync(psdns_ctx* c);
// registers tau [6][n][n][n] for the fused x pass of the next
// stage_nonlinear(kstep) of c (used once; any call that overwrites the work
// arrays or shifts drops it)
int ctx_set_stress(psdns_ctx* c, const float* tau, int kstep);
// sets the thread's last-error message and returns code
int set_error(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

namespace sgs {

constexpr int kLam = 5, kConv = 16, kHid = 64, kBasis = 4, kTaps = 27;
constexpr int kIn0 = kLam * kTaps;  // conv inputs per point
constexpr int kIn1 = kLam + kConv;  // first MLP layer inputs
constexpr int kParams = kConv * kIn0 + kConv + kHid * kIn1 + kHid + 2 * (kHid * kHid + kHid) + kBasis * kHid + kBasis;
constexpr double kQeps = 1e-30;     // floor of q = |S|^2 + |W|^2
constexpr int kMaxBatch = 65536;

// work-groups of a training step's gradient kernel = partial rows of kParams
// floats: one per tile of 64 points up to one per CU (its LDS fills a CU, and
// more rows would only lengthen the fold)
constexpr int train_rows(int B) { return (B + 63) / 64 < 256 ? (B + 63) / 64 : 256; }

// r = 2, 4, .., 32 (the ratios of two grids between 32 and 1024); -1 for another
int launch_box_filter(hipStream_t st, int prec, const void* u, int n, int r, void* ubar, float* tau);
void launch_invariants(hipStream_t st, int prec, const void* A, size_t P, double delta2, float* lam, float* T);
// the closure's stress of the features: the convolution in FP32, the dense
// layers in FP32 or on bf16 operands
void launch_predict(hipStream_t st, bool bf16, const float* lam, const float* T, int n, const float* theta, float* tau);
void launch_add_stress(hipStream_t st, int prec, void* ux, const float* tau, size_t P);
int field_err_blocks();
void launch_field_err(hipStream_t st, const float* tp, const float* tt, size_t P, double* part);
void launch_target_norm(hipStream_t st, const float* tau_s, size_t P, int nsnap, double* part);
void launch_train_batch(hipStream_t st, float* theta, const float* lam_s, const float* T_s, const float* tau_s, int n,
                        int nsnap, uint64_t base, int B, float inv, float* part, double* lpart, double scale,
                        float* grad, double* loss, float* m, float* v, float lr, long long t);

}  // namespace sgs
}  // namespace psdns
