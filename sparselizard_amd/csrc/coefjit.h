// Per-program coefficient kernels: the coefficient program of a bucket
// compiled at plan creation into straight-line device code (one thread per
// (element, Gauss point), values in registers), in place of the interpreter;
// the generated source is the prelude of build-time inlined headers
// (gen_jit_prelude.py) plus one statement per program instruction.
#pragma once
#include <hip/hip_runtime.h>
#include <string>
#include <vector>
#include "kernels/device.h"
#include "kernels/tile.h"

namespace slx {

// form functions per field at most for a per-element gather of its values
#define SLX_JIT_GATHER_NFF 16

// Record layout of a bucket's coefficients (row-wise assembly): slot s of
// element e at e * erec + pos[s] (pos < 0: not stored), zeros at the pads.
struct CoefPack {
    int erec = 0;  // 0: the [slot][point][element] layouts
    std::vector<int> pos, pads;
};

// Shape of an element kernel: the slices of a bucket whose element matrices one
// thread can hold.
struct ElemShape {
    struct Slice {
        int n_tf, n_dof;              // n_dof 0: right-hand side
        bool vec4;                    // rows start 16-byte aligned (FP32)
        std::vector<slx_term> terms;
    };
    std::vector<Slice> slices;        // every slice of the bucket
    bool affine = false, q_inv = false;
    bool store = false;               // also writes the coefficient table [slot][point][element]
};
#define SLX_ELEM_MAX 72               // element-matrix entries of one thread

// Full source of the kernel of one program (prelude included).  runs: each
// thread walks a run of Gauss points of one element (Gauss-point-varying
// buckets), and gathers the values of every field of at most
// SLX_JIT_GATHER_NFF form functions (field_nff[f] in this bucket) once for
// the run; otherwise one thread per (element, Gauss point).  With a pack
// (coefficients constant over the Gauss points) the kernel writes records.
// several: the kernel of a launch over several buckets.
std::string coef_kernel_source(const slx_instr* prog, int n_instr, bool fp64, bool runs, const std::vector<int>& field_nff,
                               const CoefPack& pack = CoefPack(), bool several = false, bool affine = false);
// Source of the element kernel slx_elem of one program: one thread per element
// evaluates the geometry, the program and the contraction of every slice, point
// by point, so that no coefficient goes through memory.
std::string elem_kernel_source(const slx_instr* prog, int n_instr, bool fp64, const std::vector<int>& field_nff, const ElemShape& shape,
                               bool several);
// Compiles (or finds in the process-wide cache) the kernel of one program for
// the current device; fp64 selects FP64 coefficients.  On failure returns
// false with the compiler log in *err.
bool coef_compile(const slx_instr* prog, int n_instr, bool fp64, bool runs, const std::vector<int>& field_nff, hipFunction_t* fn,
                  std::string* err, const CoefPack& pack = CoefPack(), bool several = false,
                  bool affine = false);
bool elem_compile(const slx_instr* prog, int n_instr, bool fp64, const std::vector<int>& field_nff, const ElemShape& shape, bool several,
                  hipFunction_t* fn, std::string* err);
hipError_t elem_launch(hipFunction_t fn, const DevBucket& b, int64_t coff, const DevJob* jobs, int n_jobs, int max_elem, const DevInputs& in,
                       void* cbase, void* ke, hipStream_t st);
// Same launch contract as the interpreter's coefficient kernel.
hipError_t coef_launch(hipFunction_t fn, const DevBucket& b, int64_t coff, const DevJob* jobs, int n_jobs, int max_elem, const DevInputs& in, int nq,
                       int qfast, void* cbase, hipStream_t st);

// One slice's tile kernel (kernels/tile_jit.h).
struct TileSpec {
    int arith;                        // 0 FP16 split, 1 BF16 split, 2 FP32
    int na, nkc, ngp, mtt, ntt, n_tf, n_dof;
    int n_store;                      // columns stored: n_dof, or more where the rows' padding may be written
    std::vector<int> term_a, term_b, term_slot;  // index of the tf derivative, dof derivative, coefficient slot
    bool several;
};
struct TileKernel {
    hipFunction_t fn = nullptr;
    int waves = 0, groups = 0;        // waves of a workgroup, workgroups on a CU
    int batch = 1;                    // elements whose coefficients a wave loads at once
};
// Source of the kernel and its launch shape; empty when its tables don't fit.
std::string tile_kernel_source(const TileSpec& spec, TileKernel& k);
bool tile_compile(const TileSpec& spec, TileKernel* k, std::string* err);
hipError_t tile_launch(const TileKernel& k, const TileJob& one, const TileJob* jobs, int n_jobs, int max_elem, const void* cbase, int qfast, float* ke,
                       int n_cu, hipStream_t st);

}  // namespace slx
