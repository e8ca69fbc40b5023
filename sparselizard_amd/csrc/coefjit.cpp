// Per-program coefficient kernels compiled with hipRTC.
//
// The interpreter (assemble.hip, run_program) keeps its register file in
// per-lane scratch memory, so every instruction waits on a memory round trip.
// Here the program of a bucket becomes one straight-line kernel: each
// instruction is a statement on a fresh value (static single assignment), the
// compiler keeps the values in VGPRs, and the program's arithmetic is the
// interpreter's, in the same order and precision (no contraction into FMAs).
// Geometry and field interpolation are the shared device helpers of
// kernels/coef_device.h, compiled with the library's flags; the compiler may
// contract them differently in the two kernels, so coefficients agree to
// rounding (measured: 1e-16 relative in FP64, 5e-8 in FP32), not bitwise.
// Kernels are cached per (device, source) for the life of the process.
#include "coefjit.h"
#include <hip/hiprtc.h>
#include <cstdio>
#include <algorithm>
#include <functional>
#include <map>
#include <mutex>
#include <sstream>
#include <vector>

#include "jit_prelude.inc"

namespace slx {
namespace {

std::mutex g_mu;
std::map<std::string, hipFunction_t> g_cache;  // key: device id + source

// One statement per program instruction; out(slot, expression) takes the
// values of SLX_OP_OUT (to be multiplied by adet).
void emit_program(std::ostringstream& o, const slx_instr* prog, int n, const std::function<int(int)>& nff_of,
                  const std::function<void(int, const std::string&)>& out) {
    std::vector<std::string> cur(SLX_MAX_PROG_REGS, "(T)0");
    for (int pc = 0; pc < n; pc++) {
        const slx_instr& x = prog[pc];
        const std::string a = (x.a >= 0 && x.a < SLX_MAX_PROG_REGS) ? cur[x.a] : "(T)0";
        const std::string bb = (x.b >= 0 && x.b < SLX_MAX_PROG_REGS) ? cur[x.b] : "(T)0";
        const std::string v = "v" + std::to_string(pc);
        std::string rhs;
        switch (x.op) {
            case SLX_OP_CONST: rhs = "(T)in.consts[" + std::to_string(x.imm) + "]"; break;
            case SLX_OP_PARAM:
                rhs = "(T)in.params[(size_t)" + std::to_string(x.imm) + " * in.param_len + ((const SLX_GLOBAL int*)b.elem_ids)[e]]";
                break;
            case SLX_OP_JAC: rhs = "(T)g.J[" + std::to_string(3 * x.a + x.b) + "]"; break;
            case SLX_OP_INVJAC: rhs = "(T)g.inv[" + std::to_string(3 * x.a + x.b) + "]"; break;
            case SLX_OP_DETJ: rhs = "(T)g.det"; break;
            case SLX_OP_COORD:
                o << "        T " << v << ";\n        {\n            double s = 0.0;\n"
                  << "            for (int k = 0; k < b.n_geo; k++) {\n"
                  << "                const int node = ((const SLX_GLOBAL int*)b.geo_nodes)[(size_t)e * b.n_geo + k];\n"
                  << "                s += in.xyz[3 * (size_t)node + " << x.a << "] * ((const SLX_CONST double*)b.geo_tab)[(size_t)k * b.n_gp + q];\n"
                  << "            }\n            " << v << " = (T)s;\n        }\n";
                cur[x.dst] = v;
                continue;
            case SLX_OP_FIELD:
                if (nff_of(x.imm) > 0)
                    rhs = "(T)field_value_pre<" + std::to_string(nff_of(x.imm)) + ">(b, " + std::to_string(x.imm) + ", fv" +
                          std::to_string(x.imm) + ", fo" + std::to_string(x.imm) + ", " + std::to_string(x.a) + ", q, g)";
                else
                    rhs = "(T)field_value(b, in, " + std::to_string(x.imm) + ", " + std::to_string(x.a) + ", e, q, g)";
                break;
            case SLX_OP_ADD: rhs = a + " + " + bb; break;
            case SLX_OP_MUL: rhs = a + " * " + bb; break;
            case SLX_OP_POW: rhs = "pow(" + a + ", " + bb + ")"; break;
            case SLX_OP_OUT:
                out(x.imm, a);
                continue;
            default: rhs = "apply_unary<T>(" + std::to_string(x.op) + ", " + a + ")"; break;
        }
        o << "        const T " << v << " = " << rhs << ";\n";
        if (x.dst >= 0 && x.dst < SLX_MAX_PROG_REGS) cur[x.dst] = v;
    }
}

// Fields whose values a thread gathers once per element (at most
// SLX_JIT_GATHER_NFF form functions).
std::vector<int> gathered_fields(const slx_instr* prog, int n, const std::vector<int>& field_nff) {
    std::vector<int> pre;
    for (int pc = 0; pc < n; pc++)
        if (prog[pc].op == SLX_OP_FIELD) {
            const int f = prog[pc].imm;
            if (f >= 0 && f < (int)field_nff.size() && field_nff[f] > 0 && field_nff[f] <= SLX_JIT_GATHER_NFF &&
                std::find(pre.begin(), pre.end(), f) == pre.end())
                pre.push_back(f);
        }
    return pre;
}

void emit_gather(std::ostringstream& o, const std::vector<int>& pre, const std::vector<int>& field_nff) {
    for (int f : pre)
        o << "    double fv" << f << "[" << field_nff[f] << "];\n    bool fo" << f << "[" << field_nff[f] << "];\n"
          << "    field_gather<" << field_nff[f] << ">(b, in, " << f << ", e, fv" << f << ", fo" << f << ");\n";
}

}  // namespace

std::string coef_kernel_source(const slx_instr* prog, int n, bool fp64, bool runs, const std::vector<int>& field_nff,
                               const CoefPack& pack, bool several, bool affine) {
    std::ostringstream o;
    // fields whose values a thread gathers once per element (runs of Gauss
    // points, at most SLX_JIT_GATHER_NFF form functions)
    const std::vector<int> pre = runs ? gathered_fields(prog, n, field_nff) : std::vector<int>();
    auto nff_of = [&](int f) { return std::find(pre.begin(), pre.end(), f) == pre.end() ? 0 : field_nff[f]; };
    o << "namespace slx {\ntypedef " << (fp64 ? "double" : "float") << " T;\n";
    // runs: one thread per (element, run of qc Gauss points).  Gauss point
    // fastest layout (qfast): qc = 1 and consecutive threads take consecutive
    // points of one element.  Element fastest layout: consecutive threads take
    // consecutive elements at the same points, each thread loads its element's
    // nodes once and walks its qc points.  Without runs (one point per element
    // or per thread): the (element, Gauss point) of the thread, qc unused.
    // several: blockIdx.y names the bucket; a single one comes by value
    o << "extern \"C\" __global__ void __launch_bounds__(256) slx_coef(" << (several ? "const DevJob* __restrict__ jobs" : "DevJob job")
      << ", DevInputs in, int nq, int qfast, int qc, unsigned char* __restrict__ cbase) {\n"
      << (several ? "    const DevJob& job = jobs[blockIdx.y];\n" : "")
      << "    const DevBucket& b = job.b;\n"
         "    T* ctab = (T*)(cbase + job.coff);\n";
    if (runs)
        o << "    const int nch = qfast ? nq : (nq + qc - 1) / qc;\n"
             "    const int64_t total = (int64_t)b.n_elem * nch;\n"
             "    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;\n"
             "    if (idx >= total) return;\n"
             "    const int e = qfast ? (int)(idx / nq) : (int)(idx % b.n_elem);\n"
             "    const int q0 = qfast ? (int)(idx % nq) : (int)(idx / b.n_elem) * qc;\n"
             "    const int q1 = qfast ? q0 + 1 : min(nq, q0 + qc);\n"
             "    GeoX gx;\n"
             "    geo_load(b, in.xyz, e, gx);\n";
    emit_gather(o, pre, field_nff);
    if (runs)
        // affine elements: one geometry for all points
        o << "    const int64_t stride = (int64_t)nq * b.n_elem;\n"
          << (affine ? "    Geo g;\n    geo_eval(b, gx, 0, g);\n" : "")
          << "    for (int q = q0; q < q1; q++) {\n"
          << (affine ? "" : "    Geo g;\n    geo_eval(b, gx, q, g);\n");
    else
        o << "    const int64_t total = (int64_t)b.n_elem * nq;\n"
             "    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;\n"
             "    if (idx >= total) return;\n"
             "    const int e = qfast ? (int)(idx / nq) : (int)(idx % b.n_elem);\n"
             "    const int q = qfast ? (int)(idx % nq) : (int)(idx / b.n_elem);\n"
             "    const int64_t stride = (int64_t)nq * b.n_elem;\n"
             "    {\n"
             "    Geo g;\n"
             "    geometry(b, in.xyz, e, q, g);\n";
    o << "    const size_t oi = qfast ? (size_t)e * nq + q : (size_t)q * b.n_elem + e;\n"
         "    const T adet = (T)fabs(g.det);\n"
         "    {\n"
         "#pragma clang fp contract(off)\n";
    // records: 16-byte stores, each as soon as its entries are known
    const int vw = fp64 ? 2 : 4;
    std::vector<std::string> rec(pack.erec);
    std::vector<int> open(pack.erec / vw + 1, vw);
    auto put = [&](int k, const std::string& v) {
        rec[k] = v;
        if (--open[k / vw] > 0) return;
        const int k0 = k / vw * vw;
        o << "        *(" << (fp64 ? "double2" : "float4") << "*)(ctab + (size_t)e * " << pack.erec << " + " << k0 << ") = "
          << (fp64 ? "make_double2(" : "make_float4(");
        for (int c = 0; c < vw; c++) o << (c ? ", " : "") << rec[k0 + c];
        o << ");\n";
    };
    for (int k : pack.pads) put(k, "(T)0");
    emit_program(o, prog, n, nff_of, [&](int slot, const std::string& v) {
        if (pack.erec > 0) {
            if (pack.pos[slot] >= 0) put(pack.pos[slot], v + " * adet");
        } else {
            o << "        ctab[(size_t)" << slot << " * stride + oi] = " << v << " * adet;\n";
        }
    });
    o << "    }\n    }\n}\n}  // namespace slx\n";
    return std::string(kJitPrelude) + o.str();
}

static bool compile_source(const std::string& src, const char* name, hipFunction_t* fn, std::string* err) {
    *fn = nullptr;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        if (err) *err = "no current device";
        return false;
    }
    const std::string key = std::to_string(dev) + "\n" + src;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_cache.find(key);
        if (it != g_cache.end()) {
            *fn = it->second;
            return true;
        }
    }
    hiprtcProgram rp;
    if (hiprtcCreateProgram(&rp, src.c_str(), "slx_coef.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS) {
        if (err) *err = "hiprtcCreateProgram failed";
        return false;
    }
    // the library's own device flags (packed FP32 instructions disabled)
    const char* opts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=fast",
                          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
    const hiprtcResult cr = hiprtcCompileProgram(rp, (int)(sizeof(opts) / sizeof(opts[0])), opts);
    if (cr != HIPRTC_SUCCESS) {
        size_t ls = 0;
        hiprtcGetProgramLogSize(rp, &ls);
        std::string log(ls + 1, '\0');
        if (ls) hiprtcGetProgramLog(rp, &log[0]);
        if (err) *err = std::string("hiprtcCompileProgram: ") + hiprtcGetErrorString(cr) + "\n" + log;
        hiprtcDestroyProgram(&rp);
        return false;
    }
    size_t cs = 0;
    hiprtcGetCodeSize(rp, &cs);
    std::vector<char> code(cs);
    hiprtcGetCode(rp, code.data());
    hiprtcDestroyProgram(&rp);
    hipModule_t mod;
    hipError_t e = hipModuleLoadData(&mod, code.data());
    if (e != hipSuccess) {
        if (err) *err = std::string("hipModuleLoadData: ") + hipGetErrorString(e);
        return false;
    }
    hipFunction_t f;
    e = hipModuleGetFunction(&f, mod, name);
    if (e != hipSuccess) {
        if (err) *err = std::string("hipModuleGetFunction: ") + hipGetErrorString(e);
        return false;
    }
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_cache.find(key);
    if (it != g_cache.end()) {
        *fn = it->second;  // compiled meanwhile by another thread; keep the first
        return true;
    }
    g_cache[key] = f;
    *fn = f;
    return true;
}

bool coef_compile(const slx_instr* prog, int n_instr, bool fp64, bool runs, const std::vector<int>& field_nff, hipFunction_t* fn,
                  std::string* err, const CoefPack& pack, bool several, bool affine) {
    return compile_source(coef_kernel_source(prog, n_instr, fp64, runs, field_nff, pack, several, affine), "slx_coef", fn, err);
}

// What bounds it: the vector ALU (FP64 geometry and fields, then the
// contraction's multiply-adds on table values in scalar registers); the
// element's matrices stay in registers and go out in 16-byte stores.  2D P2
// Newton (5e5 triangles, 12 points, 6 x 6 and a right-hand side): 0.12 ms, the
// program (0.22 ms) and element kernel (0.29 ms) with the 144 MB coefficient
// table between them before.
std::string elem_kernel_source(const slx_instr* prog, int n, bool fp64, const std::vector<int>& field_nff, const ElemShape& shape,
                               bool several) {
    std::ostringstream o;
    const std::vector<int> pre = gathered_fields(prog, n, field_nff);
    auto nff_of = [&](int f) { return std::find(pre.begin(), pre.end(), f) == pre.end() ? 0 : field_nff[f]; };
    o << "namespace slx {\ntypedef " << (fp64 ? "double" : "float") << " T;\n";
    o << "extern \"C\" __global__ void __launch_bounds__(256) slx_elem(" << (several ? "const DevJob* __restrict__ jobs" : "DevJob job")
      << ", DevInputs in, unsigned char* __restrict__ cbase, T* __restrict__ ke) {\n"
      << (several ? "    const DevJob& job = jobs[blockIdx.y];\n" : "")
      << "    const DevBucket& b = job.b;\n"
         "    const int e = (int)(blockIdx.x * 256 + threadIdx.x);\n"
         "    if (e >= b.n_elem) return;\n"
         "    GeoX gx;\n"
         "    geo_load(b, in.xyz, e, gx);\n";
    if (shape.store) o << "    T* ctab = (T*)(cbase + job.coff);\n";
    emit_gather(o, pre, field_nff);
    o << "    const int ngp = b.n_gp;\n"
         "    const SLX_CONST double* gw = (const SLX_CONST double*)b.gp_w;\n";
    const char* sfx = fp64 ? "" : "32";
    for (size_t k = 0; k < shape.slices.size(); k++) {
        const auto& sl = shape.slices[k];
        o << "    const SLX_CONST T* tf" << k << " = (const SLX_CONST T*)b.slices[" << k << "].tf_tabq" << sfx << ";\n"
          << "    const int tp" << k << " = b.slices[" << k << "].tf_pad;\n";
        if (sl.n_dof > 0)
            o << "    const SLX_CONST T* df" << k << " = (const SLX_CONST T*)b.slices[" << k << "].dof_tabq" << sfx << ";\n"
              << "    const int dp" << k << " = b.slices[" << k << "].dof_pad;\n";
        o << "    T acc" << k << "[" << sl.n_tf * std::max(sl.n_dof, 1) << "] = {};\n";
    }
    int n_coefs = 0;
    for (int pc = 0; pc < n; pc++)
        if (prog[pc].op == SLX_OP_OUT) n_coefs = std::max(n_coefs, prog[pc].imm + 1);
    for (int c = 0; c < n_coefs; c++) o << "    T c" << c << " = (T)0;\n";
    // the program, once for all points where nothing depends on the point
    auto program = [&](const char* q, const char* stride, const char* at) {
        o << "        const T adet = (T)fabs(g.det);\n        {\n#pragma clang fp contract(off)\n        const int q = " << q << ";\n";
        emit_program(o, prog, n, nff_of, [&](int slot, const std::string& v) { o << "        c" << slot << " = " << v << " * adet;\n"; });
        o << "        }\n";
        if (shape.store)
            for (int c = 0; c < n_coefs; c++) o << "        ctab[(size_t)" << c << " * " << stride << " + " << at << "] = c" << c << ";\n";
    };
    if (shape.affine || shape.q_inv) o << "    Geo g;\n    geo_eval(b, gx, 0, g);\n";
    if (shape.q_inv) {
        o << "    {\n";
        program("0", "b.n_elem", "e");
        o << "    }\n";
    }
    o << "    for (int qq = 0; qq < ngp; qq++) {\n";
    if (!shape.q_inv) {
        if (!shape.affine) o << "        Geo g;\n        geo_eval(b, gx, qq, g);\n";
        program("qq", "((int64_t)ngp * b.n_elem)", "(size_t)qq * b.n_elem + e");
    }
    o << "        const T w = (T)gw[qq];\n";
    for (size_t k = 0; k < shape.slices.size(); k++) {
        const auto& sl = shape.slices[k];
        for (int r = 0; r < 4; r++) {
            std::vector<const slx_term*> ts;
            for (const slx_term& t : sl.terms)
                if (t.tf_deriv == r) ts.push_back(&t);
            if (ts.empty()) continue;
            o << "        {\n            const SLX_CONST T* tv = tf" << k << " + ((size_t)qq * 4 + " << r << ") * tp" << k << ";\n";
            if (sl.n_dof == 0) {
                o << "            const T h = w * (";
                for (size_t t = 0; t < ts.size(); t++) o << (t ? " + " : "") << "c" << ts[t]->coef;
                o << ");\n#pragma unroll\n            for (int i = 0; i < " << sl.n_tf << "; i++) acc" << k << "[i] += tv[i] * h;\n";
            } else {
                o << "            const SLX_CONST T* dv = df" << k << " + (size_t)qq * 4 * dp" << k << ";\n"
                  << "            T h[" << sl.n_dof << "];\n#pragma unroll\n            for (int j = 0; j < " << sl.n_dof << "; j++) h[j] = w * (";
                for (size_t t = 0; t < ts.size(); t++)
                    o << (t ? " + " : "") << "c" << ts[t]->coef << " * dv[" << ts[t]->dof_deriv << " * dp" << k << " + j]";
                o << ");\n#pragma unroll\n            for (int i = 0; i < " << sl.n_tf << "; i++) {\n                const T t = tv[i];\n"
                  << "#pragma unroll\n                for (int j = 0; j < " << sl.n_dof << "; j++) acc" << k << "[i * " << sl.n_dof
                  << " + j] += t * h[j];\n            }\n";
            }
            o << "        }\n";
        }
    }
    o << "    }\n";
    for (size_t k = 0; k < shape.slices.size(); k++) {
        const auto& sl = shape.slices[k];
        o << "    {\n        T* out = ke + b.slices[" << k << "].ke_base + (int64_t)e * " << sl.n_tf << " * b.slices[" << k << "].ke_ld;\n"
          << "        const int64_t ld = b.slices[" << k << "].ke_ld;\n";
        if (sl.n_dof == 0) {
            o << "#pragma unroll\n        for (int i = 0; i < " << sl.n_tf << "; i++) out[i * ld] = -acc" << k << "[i];\n";
        } else {
            o << "#pragma unroll\n        for (int i = 0; i < " << sl.n_tf << "; i++) {\n";
            const int vw = fp64 ? 2 : 4;
            int j = 0;
            if (sl.vec4)
                for (; j + vw <= sl.n_dof; j += vw) {
                    o << "            *(" << (fp64 ? "double2" : "float4") << "*)(out + i * ld + " << j << ") = " << (fp64 ? "make_double2(" : "make_float4(");
                    for (int c = 0; c < vw; c++) o << (c ? ", " : "") << "acc" << k << "[i * " << sl.n_dof << " + " << j + c << "]";
                    o << ");\n";
                }
            for (; j < sl.n_dof; j++) o << "            out[i * ld + " << j << "] = acc" << k << "[i * " << sl.n_dof << " + " << j << "];\n";
            o << "        }\n";
        }
        o << "    }\n";
    }
    o << "}\n}  // namespace slx\n";
    return std::string(kJitPrelude) + o.str();
}

bool elem_compile(const slx_instr* prog, int n_instr, bool fp64, const std::vector<int>& field_nff, const ElemShape& shape, bool several,
                  hipFunction_t* fn, std::string* err) {
    return compile_source(elem_kernel_source(prog, n_instr, fp64, field_nff, shape, several), "slx_elem", fn, err);
}

hipError_t elem_launch(hipFunction_t fn, const DevBucket& b, int64_t coff, const DevJob* jobs, int n_jobs, int max_elem, const DevInputs& in,
                       void* cbase, void* ke, hipStream_t st) {
    if (max_elem == 0) return hipSuccess;
    DevInputs ii = in;
    DevJob job{b, coff};
    void* args[] = {n_jobs > 1 ? (void*)&jobs : (void*)&job, &ii, &cbase, &ke};
    return hipModuleLaunchKernel(fn, (unsigned)((max_elem + 255) / 256), (unsigned)n_jobs, 1, 256, 1, 1, 0, st, args, nullptr);
}

hipError_t coef_launch(hipFunction_t fn, const DevBucket& b, int64_t coff, const DevJob* jobs, int n_jobs, int max_elem, const DevInputs& in, int nq,
                       int qfast, void* cbase, hipStream_t st) {
    const int64_t pairs = (int64_t)max_elem * nq;
    if (pairs == 0 || b.n_coefs == 0) return hipSuccess;
    // element-fastest layout: runs of qc points per thread, as long as about
    // 256K threads remain to fill the GPU
    // (a kernel compiled without runs has nq = 1 here, so qc = 1 and the grid
    // is one thread per element)
    int qc = 1;
    if (!qfast) qc = (int)std::max<int64_t>(1, std::min<int64_t>(nq, pairs * n_jobs / (256 * 1024)));
    const int64_t nch = qfast ? nq : (nq + qc - 1) / qc;
    const int64_t total = (int64_t)max_elem * nch;
    DevInputs ii = in;
    DevJob job{b, coff};
    void* args[] = {n_jobs > 1 ? (void*)&jobs : (void*)&job, &ii, &nq, &qfast, &qc, &cbase};
    return hipModuleLaunchKernel(fn, (unsigned)((total + 255) / 256), (unsigned)n_jobs, 1, 256, 1, 1, 0, st, args, nullptr);
}

// Where the tables are kept and how many waves share them.  Registers: both
// tables in at most 72 (1 x 1 tiles of up to 4 chunks), or the dof table in at most
// 40 with P in LDS: more would leave fewer than three waves a SIMD.  The
// registers that are held across the chunk loop then say how many waves a SIMD
// takes (the compiler adds about 20 to 40; measured without scratch on 16 x 16 to
// 64 x 64 slices).  LDS: as many workgroups of 4 or 8 waves as 144 KB hold (three
// 53 KB groups of a CU don't start together), or one with the whole 160 KB.
std::string tile_kernel_source(const TileSpec& s, TileKernel& k) {
    const int nt = (int)s.term_a.size();
    std::vector<int> bl, pa, pb, tp;
    for (int b = 0; b < 4; b++)
        if (std::find(s.term_b.begin(), s.term_b.end(), b) != s.term_b.end()) bl.push_back(b);
    for (int t = 0; t < nt; t++) {
        const int bi = (int)(std::find(bl.begin(), bl.end(), s.term_b[t]) - bl.begin());
        int x = 0;
        while (x < (int)pa.size() && (pa[x] != s.term_a[t] || pb[x] != bi)) x++;
        if (x == (int)pa.size()) {
            pa.push_back(s.term_a[t]);
            pb.push_back(bi);
        }
        tp.push_back(x);
    }
    const int nb = (int)bl.size(), np = (int)pa.size(), qh = 8 / s.na, ngpp = s.nkc * 4 * qh, npl = s.arith == 1 ? 3 : 2;
    const int hregs = s.nkc * s.ntt * qh * nb, pregs = s.nkc * s.mtt * npl * 4;
    const bool preg = hregs + pregs <= 72, hreg = preg || hregs <= 40;
    // four elements' coefficients at a time where they fit the registers and their
    // rows the LDS beside eight waves' tables
    const int cregs = (ngpp + 63) / 64 * nt;
    const size_t tables = (size_t)(hreg ? 0 : hregs * 256) + (size_t)(preg ? 0 : pregs * 256), row = (size_t)np * ngpp * 4;
    k.batch = cregs <= 9 && tables + 32 * row <= 72 * 1024 ? 4 : 1;
    const int held = (preg ? pregs : s.mtt * npl * 4) + (hreg ? hregs : qh * nb) + s.mtt * s.ntt * 4 + npl * 4 + np * qh;
    const int occ = held <= 110 ? 4 : held <= 124 ? 3 : 2;
    const size_t wave = k.batch * row;
    k.waves = 0;
    for (int w : {4, 8}) {
        const size_t need = tables + w * wave;
        const int g = std::min<int>(4 * occ / w, (int)(144 * 1024 / need));
        if (g >= 1 && w * g > k.waves * k.groups) {
            k.waves = w;
            k.groups = g;
        }
    }
    if (k.waves * k.groups < 8 && tables + 8 * wave <= 160 * 1024) {
        k.waves = 8;
        k.groups = 1;
    }
    if (k.waves == 0) return std::string();
    std::ostringstream o;
    auto list = [&](const char* name, const std::vector<int>& v) {
        o << "constexpr int " << name << "[] = {";
        for (size_t i = 0; i < v.size(); i++) o << (i ? ", " : "") << v[i];
        o << "};\n";
    };
    o << "#define TJ_ARG " << (s.several ? "const TileJob* __restrict__ jobs" : "TileJob job") << "\n#define TJ_JOB "
      << (s.several ? "const TileJob& job = jobs[blockIdx.y]" : "") << "\nnamespace slx { namespace tj {\nconstexpr int AR = " << s.arith
      << ", NA = " << s.na << ", NB = " << nb << ", NT = " << nt << ", NP = " << np << ", NKC = " << s.nkc << ", NGP = " << s.ngp << ", MTT = " << s.mtt
      << ", NTT = " << s.ntt << ", N_TF = " << s.n_tf << ", N_STORE = " << s.n_store << ", EB = " << k.batch << ", WAVES = " << k.waves
      << ", OCC = " << occ << ";\nconstexpr bool H_REG = " << (hreg ? "true" : "false") << ", P_REG = " << (preg ? "true" : "false") << ";\n";
    list("B_OF", bl);
    list("PAIR_A", pa);
    list("PAIR_B", pb);
    list("TERM_PAIR", tp);
    list("TERM_SLOT", s.term_slot);
    o << "} }\n";
    return std::string(kTilePrelude) + o.str() + kTileKernel;
}

bool tile_compile(const TileSpec& s, TileKernel* k, std::string* err) {
    const std::string src = tile_kernel_source(s, *k);
    k->fn = nullptr;
    if (src.empty()) return false;  // the tables exceed the LDS
    return compile_source(src, "slx_tile", &k->fn, err);
}

hipError_t tile_launch(const TileKernel& k, const TileJob& one, const TileJob* jobs, int n_jobs, int max_elem, const void* cbase, int qfast, float* ke,
                       int n_cu, hipStream_t st) {
    if (max_elem == 0 || n_jobs == 0) return hipSuccess;
    TileJob job = one;
    void* args[] = {n_jobs > 1 ? (void*)&jobs : (void*)&job, &cbase, &qfast, &ke};
    const int step = k.waves * k.batch;
    const int64_t groups = ((int64_t)max_elem + step - 1) / step, fit = ((int64_t)n_cu * k.groups + n_jobs - 1) / n_jobs;
    return hipModuleLaunchKernel(k.fn, (unsigned)((std::min(groups, fit) + 7) / 8 * 8), (unsigned)n_jobs, 1, 64 * k.waves, 1, 1, 0, st, args, nullptr);
}

}  // namespace slx
