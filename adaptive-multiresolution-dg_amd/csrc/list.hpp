// Source lists of the 1D sweeps and the kernels that run on them
// (list_kern.hip); the stage built from them is in list_stage.hip.
//
// A sweep along dimension d sums, for every target element, over the related
// present cells of its d-fiber in ascending slot order.  The lists hold those
// cells, found once per grid change instead of once per sweep (a stage runs
// tens of sweeps and a time step four stages): per target the source elements
// in that order, first the ones at levels up to the target's own (the U
// part), then the finer ones (the L part).  A pair whose block of the sweep's
// table is entirely zero is left out: the products it would add are zeros,
// and a sum that starts at +0 never is -0, so no value changes.  What is left
// out is most of the descendants of the coarse targets: a point of a coarse
// cell lies in one cell per finer level, and an interface touches two.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kern.hpp"

namespace adg {

// Kinds of lists, by relation and table: point values of the Alpert basis,
// volume tables (u_v, u_vx; no zero blocks), flux and penalty tables, and the
// assembled constant-coefficient operator.
enum ListKind { LIST_PT = 0, LIST_VOL, LIST_FLX, LIST_LIN, LIST_KINDS };

// One 1D sweep over a list; plain data in device memory, read through scalar
// loads (the term is the same for a whole wavefront).
struct ListTerm {
  const double* in;   // null: the stage's current coefficients (kernel argument u)
  const float* in32;  // FP32 form: input in FP32 (null: in or u, rounded on load)
  const double* M;
  const float *Mh, *Ml;  // FP32 form: the table as the sum of two FP32 parts
  // per element: first entry, number of U entries | all entries << 16, slot
  // in the swept dimension, instance
  const int4* meta;
  const int2* ent;   // source element, source slot
  const int2* rofs;  // per rest index: offsets into the input and output tensor
  const double* coef_inst;  // per-instance coefficient (replaces coef when non-null)
  void* out;                // phase terms: output buffer
  double coef;
  int comp;  // component of the input: it starts comp * E * comp_size values in
  int comp_size;
  int Tin, Tout, sdd, sod, R, ns, lu;
};

// ---- list build ----
struct ListBuildArgs {
  const int32_t* slot[kMaxDimK];
  const int32_t* fbase[kMaxDimK];
  const int32_t* fmaxl[kMaxDimK];
  const int32_t* fmap[kMaxDimK];
  const uint32_t* fbits[kMaxDimK];
  const int32_t* lsum;
  const int32_t* inst;
  // pairs of each kind: rows of ns bits (whole words) per target slot
  const uint32_t* nz[LIST_KINDS];
  int4* meta[LIST_KINDS * kMaxDimK];  // [kind * D + d]; null: not built
  int2* ent[LIST_KINDS * kMaxDimK];
  int64_t cap[LIST_KINDS * kMaxDimK];  // entries that fit
  int32_t* total;                      // [LIST_KINDS * D], zeroed
  int32_t* err;
  int64_t E;
  int D, ns, level_cap;
};
void list_fill_totals(int32_t* total, int n, hipStream_t s);  // zeroes the counters
// lmax: deepest level of the grid in any dimension
void list_build(const ListBuildArgs& a, int kind0, int nkind, int lmax, hipStream_t s);
// sets the bit of every pair whose block of M is not zero (no M: every pair),
// among nested cells only when in_support
void list_nonzero(uint32_t* nz, const double* M, int ns, int block, bool in_support, bool clear, hipStream_t s);

// ---- sweeps ----
// term values of a block of a final kernel, kept in LDS
constexpr int kFinalValues = 65536 / 8;
template <class T>
void list_phase(int pf1, int pt1, const ListTerm* terms, int ntask, int64_t E, int R, const double* u, hipStream_t s);
template <class T>
void list_up_final(int k1, int m1, const ListTerm* terms, int nterm, int64_t E, int P, const double* u, T* up, T* fp, const double* vcoef, int kind, double fs, int ncomp, hipStream_t s);
// What the last sweeps of a right-hand side end in.
struct ListRhs {
  double* rhs;
  int add;            // 1: the terms are added to rhs, 0: it is replaced
  const double* u;    // current coefficients
  double* u_next;     // RK stage update (null: the right-hand side alone)
  const double* tn;   // u^n
  double* tn_store;   // null, or where a step's first stage keeps u^n (tn is u then)
  int scheme, stage;
  double dt;
  const double* dtv;  // per-instance step sizes (null: dt)
  int32_t* err;
  double coef[kMaxDimK];  // coefficients of the npen last terms (their own are not read)
};
// nterm terms of m1 x k1 blocks, then npen of k1 x k1 blocks on the coefficients
template <class T>
void list_rhs_final(int m1, int k1, const ListTerm* terms, int nterm, int npen, int64_t E, int K, const ListRhs& r,
                    hipStream_t s);

}  // namespace adg
