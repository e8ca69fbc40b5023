// Row-wise assembly of element matrices whose coefficients are constant over
// the Gauss points (direct.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "device.h"

namespace slx {

#define SLX_DIRECT_MAXB 3       // slices (dof fields) per segment group
#define SLX_DIRECT_MAXP 12      // derivative pairs per slice
#define SLX_DIRECT_LDS (160 * 1024)      // of one workgroup, alone on its compute unit
#define SLX_DIRECT_CU_LDS (144 * 1024)   // of several workgroups on a compute unit
#define SLX_DIRECT_PHI (32 * 1024)       // largest table of Gauss-point sums, in FP64
#define SLX_DIRECT_PAD 16                // segments and slot blocks readable past the last row

// One plan's row-wise description.  A segment (element e, group a, tf function
// i) is the 32-bit word (e * na + a) << ib | i; its entries are
//   Ke(b, j) = sum_p C(e)[a][b][p] Phi_p[i][j],   b < nb, j < n_dof
// with C the element's coefficient record ([a][rec]: nb * P values rounded up to
// 4, then the group's share of the bucket's right-hand-side coefficients rounded up
// to 4; zeros in the padding) and Phi the Gauss-point sums of the table products.
struct DirectDev {
    int32_t n_tf, n_dof, na, nb;
    int32_t P, JL, G;                       // pairs rounded up to a kernel's; columns per lane, lanes per row
    int32_t ib, rec, n_cu;
    int32_t phi_row;                        // table entries per (tf function, lane)
    int32_t slot_bytes, slot_words;         // a lane's slots of one segment: slot_words 32-bit words
    const uint64_t* desc;                   // row descriptors as DevReduce::rdesc, word 3 = first segment's slot block
    const uint32_t* seg;
    const uint32_t* slots;                  // [slot block][G][slot_words]; absent entries name the row's spare accumulator
    const float* phi32;                     // [n_tf][G][phi_row]: pair p, column jj at p * JL + jj
    const double* phi64;
    // right-hand side: word e << rib | k, value -C(e)[k's slot] rphi[k]; coefficient at rbase[k] + e * rstride
    int32_t has_rhs, rib;
    int64_t rstride, nrows;
    const int64_t* rptr;                    // [nrows + 1]
    const uint32_t* rseg;
    const int64_t* rbase;
    const double* rphi;
    const int64_t* free_dofs;
};

// Segment words, per-lane slots and row descriptors from the plan's reduction maps.
struct DirectBuild {
    int64_t nrows, n_erows, n_rhs;
    const uint64_t* rdesc;
    const uint64_t* erows;
    const uint64_t* rhs_erows;
    const void* slots;
    int32_t slot_bytes, seg_len, n_elem, ld;
    int64_t group_base[8];
    int32_t n_rgroups, rn_elem;
    int64_t rgroup_base[SLX_MAX_SLICES];
    int32_t rgroup_ntf[SLX_MAX_SLICES], rgroup_k[SLX_MAX_SLICES];  // functions, first k
};

struct DirectLaunch {
    const void *ctab, *rtab;
    double *Aval, *Dval, *rhs;
    int64_t pos0, pos1;
    int len;  // longest row
    bool with_rhs;
    hipStream_t st;
};

inline size_t direct_phi_bytes(const DirectDev& d, bool fp64) {
    return ((size_t)d.n_tf * d.G * d.phi_row * (fp64 ? 8 : 4) + 15) / 16 * 16;
}

inline int direct_stride(int len) { return (len + 1) | 1; }  // the row, a spare entry, odd: rows start on different banks

bool direct_shape(DirectDev& d, int n_pairs);
hipError_t launch_direct_build(const DirectDev& d, const DirectBuild& b, uint64_t* desc, uint32_t* seg, uint32_t* slots,
                               uint32_t* rseg, hipStream_t st, const int64_t* class_begin, const int64_t* class_end, int n_classes);
// Longest row (A + D columns) the LDS accumulators hold.
int direct_max_row(const DirectDev& d);
hipError_t launch_direct(const DirectDev& d, bool fp64, const void* ctab, const void* rtab, double* Aval, double* Dval, double* rhs,
                         hipStream_t st, const int64_t* class_begin, const int64_t* class_end, const int* class_len, int n_classes);
hipError_t launch_direct_f32(const DirectDev& d, const DirectLaunch& q);
hipError_t launch_direct_f64(const DirectDev& d, const DirectLaunch& q);
// Element matrices (and right-hand-side values) of the same coefficients, in
// the plan's element-matrix layout (inspection only).
hipError_t launch_direct_ke(const DirectDev& d, const DirectBuild& b, bool fp64, const void* ctab, const void* rtab, void* ke,
                            hipStream_t st);

}  // namespace slx
