// Row-wise assembly: element-matrix entries are computed where the CSR row
// that needs them is summed, so no element matrix is written to memory.
//
// For affine elements with coefficients constant per element,
//   Ke[(a, i)][(b, j)] = sum_p C(e)[a][b][p] Phi_p[i][j],
//   Phi_p[i][j] = sum_q w_q tf_r(p)[i][q] dof_s(p)[j][q]
// (contribution.cpp:172-246 with the Gauss-point sum taken once, in FP64, when
// the plan is made).  A segment of a row needs nb * P coefficients (27 for
// elasticity, about one 128-byte line) and nb * n_dof * P multiply-adds, while
// reading it back from memory costs a 128-byte line as well and writing it
// cost another: computing it in place removes the element-matrix round trip,
// the largest part of the traffic (64^3 P2 elasticity: 5.6 GB written and 5.6
// GB read of 16 GB per assembly).
//
// G lanes own one row, each JL consecutive columns of every dof field; the
// coefficients come through the caches (a record serves the n_tf rows of its
// element, which are close in the row order; workgroups of one XCD take
// consecutive rows so that its L2 holds them), Phi from LDS with 16-byte
// reads, and the FP64 sums are LDS accumulators as in reduce_rows
// (rawmat.cpp:67-125): segments in their fixed order, no two lanes of a
// segment on one slot, so repeated runs are bitwise equal.
#include <algorithm>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include "direct.h"

namespace slx {

// ------------------------------------------------------------ plan creation --

// Segment word of an element-matrix offset.
__device__ inline uint32_t direct_word(const DirectDev& d, const DirectBuild& b, uint64_t erow) {
    const int64_t off = (int64_t)(erow & 0xFFFFFFFFFFFFull);
    int a = 0;
    while (a + 1 < d.na && off >= b.group_base[a + 1]) a++;
    const int64_t r = (off - b.group_base[a]) / b.ld;
    const int64_t e = r / d.n_tf, i = r - e * d.n_tf;
    return ((uint32_t)(e * d.na + a) << d.ib) | (uint32_t)i;
}

// Row order inside a reduction class: blocks of 4096 elements (their records
// stay in one XCD's L2), in a block by segment count (the rows of a wave end
// together), then by the first segment's element, function and group, so that
// the rows that read one record follow each other.
__global__ void direct_key_kernel(DirectDev d, DirectBuild b, int64_t pos0, int64_t pos1, int cls, uint64_t* __restrict__ key,
                                  uint32_t* __restrict__ val) {
    const int64_t pos = pos0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (pos >= pos1) return;
    const uint64_t w2 = b.rdesc[4 * pos + 2];
    const int64_t nk = (int64_t)(w2 >> 48);
    uint64_t k = 0;
    if (nk > 0) {
        const uint32_t w = direct_word(d, b, b.erows[w2 & 0xFFFFFFFFFFFFull]);
        const uint32_t ea = w >> d.ib, e = ea / d.na, a = ea - e * d.na, i = w & ((1u << d.ib) - 1u);
        k = (uint64_t)(e >> 12) << 36 | (uint64_t)(255 - min(nk, (int64_t)255)) << 28 | (uint64_t)(e & 4095u) << 16 | (uint64_t)(i * d.na + a);
    }
    key[pos] = (uint64_t)cls << 56 | k;
    val[pos] = (uint32_t)pos;
}

__global__ void direct_count_kernel(DirectBuild b, const uint32_t* __restrict__ order, int64_t* __restrict__ nk) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t <= b.nrows) nk[t] = t < b.nrows ? (int64_t)(b.rdesc[4 * (int64_t)order[t] + 2] >> 48) : 0;
}

__global__ void direct_rhs_kernel(DirectDev d, DirectBuild b, uint32_t* __restrict__ rseg) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= b.n_rhs) return;
    const int64_t off = (int64_t)(b.rhs_erows[t] & 0xFFFFFFFFFFFFull);
    int g = 0;
    while (g + 1 < b.n_rgroups && off >= b.rgroup_base[g + 1]) g++;
    const int64_t r = off - b.rgroup_base[g];
    const int64_t e = r / b.rgroup_ntf[g], i = r - e * b.rgroup_ntf[g];
    rseg[t] = ((uint32_t)e << d.rib) | (uint32_t)(b.rgroup_k[g] + i);
}

// Row descriptors, segment words and slots in the kernel's order, one thread
// per row.  Rows with identical slot blocks share one copy, as in the source
// (every sharer writes the same words).
template <typename ST>
__global__ void direct_row_kernel(DirectDev d, DirectBuild b, const uint32_t* __restrict__ order, const int64_t* __restrict__ first,
                                  uint64_t* __restrict__ desc, uint32_t* __restrict__ seg, uint32_t* __restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < SLX_DIRECT_PAD) seg[b.n_erows + t] = 0;  // read past the last row's end, never summed
    if (t >= b.nrows) return;
    const uint64_t* rd = b.rdesc + 4 * (int64_t)order[t];
    const int JL = d.JL, G = d.G, slot_words = d.slot_words, padl = (b.seg_len + 3) & ~3;
    const int64_t sb = (int64_t)rd[3] / padl, k0 = (int64_t)(rd[2] & 0xFFFFFFFFFFFFull);
    const int nk = (int)(rd[2] >> 48), per = 4 / (int)sizeof(ST);
    desc[4 * t] = rd[0];
    desc[4 * t + 1] = rd[1];
    desc[4 * t + 2] = (uint64_t)first[t] | (uint64_t)nk << 48;
    desc[4 * t + 3] = (uint64_t)sb;
    const uint32_t spare = (uint32_t)(rd[0] >> 48) + (uint32_t)(rd[1] >> 48);  // A + D columns
    const ST* src = (const ST*)b.slots + rd[3];
    for (int k = 0; k < nk; k++) {
        seg[first[t] + k] = direct_word(d, b, b.erows[k0 + k]);
        for (int l = 0; l < G; l++)
            for (int w = 0; w < slot_words; w++) {
                uint32_t word = 0;
                for (int c = 0; c < per; c++) {
                    const int x = w * per + c, f = x / JL, j = l * JL + x % JL;
                    uint32_t s = spare;
                    if (f < d.nb && j < d.n_dof) {
                        const ST v = src[(int64_t)k * padl + f * d.n_dof + j];
                        if (v != (ST)~(ST)0) s = v;
                    }
                    word |= s << (8 * (int)sizeof(ST) * c);
                }
                out[((sb + k) * G + l) * slot_words + w] = word;
            }
    }
}

hipError_t launch_direct_build(const DirectDev& d, const DirectBuild& b, uint64_t* desc, uint32_t* seg, uint32_t* slots,
                               uint32_t* rseg, hipStream_t st, const int64_t* cb, const int64_t* ce, int nc) {
    const int64_t n = b.nrows;
    const unsigned grid = (unsigned)(n / 256 + 1);
    uint64_t *k0 = nullptr, *k1 = nullptr;
    uint32_t *v0 = nullptr, *order = nullptr;
    int64_t *nk = nullptr, *first = nullptr;
    void* tmp = nullptr;
    auto run = [&]() -> hipError_t {
        hipError_t e;
        const size_t m = (size_t)n + 1;
        if ((e = hipMalloc(&k0, m * 8)) || (e = hipMalloc(&k1, m * 8)) || (e = hipMalloc(&v0, m * 4)) || (e = hipMalloc(&order, m * 4)) ||
            (e = hipMalloc(&nk, m * 8)) || (e = hipMalloc(&first, m * 8)))
            return e;
        size_t s1 = 0, s2 = 0;
        if ((e = rocprim::radix_sort_pairs(nullptr, s1, k0, k1, v0, order, (size_t)n, 0, 64, st))) return e;
        if ((e = rocprim::exclusive_scan(nullptr, s2, nk, first, int64_t(0), m, rocprim::plus<int64_t>(), st))) return e;
        if ((e = hipMalloc(&tmp, std::max<size_t>(std::max(s1, s2), 16)))) return e;
        for (int c = 0; c < nc; c++)
            if (ce[c] > cb[c])
                hipLaunchKernelGGL(direct_key_kernel, dim3((unsigned)((ce[c] - cb[c] + 255) / 256)), dim3(256), 0, st, d, b, cb[c], ce[c], c, k0, v0);
        if (n > 0 && (e = rocprim::radix_sort_pairs(tmp, s1, k0, k1, v0, order, (size_t)n, 0, 64, st))) return e;
        hipLaunchKernelGGL(direct_count_kernel, dim3(grid), dim3(256), 0, st, b, order, nk);
        if ((e = rocprim::exclusive_scan(tmp, s2, nk, first, int64_t(0), m, rocprim::plus<int64_t>(), st))) return e;
        if (b.slot_bytes == 1) hipLaunchKernelGGL((direct_row_kernel<uint8_t>), dim3(grid), dim3(256), 0, st, d, b, order, first, desc, seg, slots);
        else hipLaunchKernelGGL((direct_row_kernel<uint16_t>), dim3(grid), dim3(256), 0, st, d, b, order, first, desc, seg, slots);
        if (d.has_rhs && b.n_rhs > 0)
            hipLaunchKernelGGL(direct_rhs_kernel, dim3((unsigned)((b.n_rhs + 255) / 256)), dim3(256), 0, st, d, b, rseg);
        if ((e = hipGetLastError())) return e;
        return hipStreamSynchronize(st);
    };
    const hipError_t e = run();
    for (void* p : {(void*)k0, (void*)k1, (void*)v0, (void*)order, (void*)nk, (void*)first, tmp})
        if (p) (void)hipFree(p);
    return e;
}

// ----------------------------------------------------------------- launches --

// Pairs are rounded up to a kernel's count (zero table entries and
// coefficients).  One, two or four lanes of a quad share a row.
bool direct_shape(DirectDev& d, int n_pairs) {
    if (d.nb < 1 || d.nb > SLX_DIRECT_MAXB || n_pairs < 1 || n_pairs > SLX_DIRECT_MAXP) return false;
    if (d.nb == 2 && n_pairs > 9) return false;
    d.P = n_pairs <= 4 && d.nb < 3 ? 4 : n_pairs <= 9 ? 9 : 12;
    if (d.n_dof > 20) return false;
    d.G = d.n_dof <= 3 ? 1 : d.n_dof <= 6 ? 2 : 4;
    d.JL = d.n_dof == 4 ? 2 : d.n_dof <= 12 ? 3 : 5;
    d.phi_row = (d.P * d.JL + 3) / 4 * 4;
    return direct_phi_bytes(d, true) <= SLX_DIRECT_PHI;
}

int direct_max_row(const DirectDev& d) {
    const int64_t left = (int64_t)SLX_DIRECT_LDS - (int64_t)direct_phi_bytes(d, true);
    return (int)std::min<int64_t>(left / 8 - 2, d.G == 4 ? 65534 : 254);
}

hipError_t launch_direct(const DirectDev& d, bool fp64, const void* ctab, const void* rtab, double* Aval, double* Dval, double* rhs,
                         hipStream_t st, const int64_t* cb, const int64_t* ce, const int* cl, int nc) {
    if (d.nrows == 0) return hipSuccess;
    const size_t phi = direct_phi_bytes(d, fp64);
    for (int c = 0; c < nc;) {
        // classes whose longest row keeps eight workgroups on a CU run together;
        // so do all the rows that the waves in flight hold at once with the
        // longest one's accumulators: no wave takes a second batch then, and one
        // launch ends with its longest rows, where several add theirs up (P2
        // elasticity, us an assembly in the FP16 split, one launch against one per
        // class: 3^3 x 6 213 and 236, 8^3 x 6 42 and 65)
        int last = c;
        const size_t wave = (size_t)(64 / d.G) * direct_stride(cl[c]) * 8;
        const int64_t waves = (int64_t)std::min<size_t>(8, (SLX_DIRECT_CU_LDS - phi) / wave) * d.n_cu;
        if (4 * wave + phi <= 20 * 1024 || ce[nc - 1] - cb[c] <= waves * (64 / d.G)) last = nc - 1;
        DirectLaunch q{ctab, rtab, Aval, Dval, rhs, cb[c], ce[last], cl[c], d.has_rhs && last == nc - 1, st};
        const hipError_t e = fp64 ? launch_direct_f64(d, q) : launch_direct_f32(d, q);
        if (e != hipSuccess) return e;
        c = last + 1;
    }
    return hipSuccess;
}

// One thread per element-matrix entry, the sums of direct_rows.
template <typename KT>
__global__ void direct_ke_kernel(DirectDev d, DirectBuild b, const KT* __restrict__ ctab, const KT* __restrict__ rtab, KT* __restrict__ ke) {
    const KT* phi;
    if constexpr (sizeof(KT) == 4) phi = (const KT*)d.phi32;
    else phi = (const KT*)d.phi64;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int per = d.nb * d.n_dof;
    const int64_t nmat = (int64_t)d.na * b.n_elem * d.n_tf * per;
    if (t < nmat) {
        const int x = (int)(t % per), f = x / d.n_dof, j = x - f * d.n_dof;
        const int64_t r = t / per;  // (a, e, i)
        const int i = (int)(r % d.n_tf), a = (int)(r / d.n_tf / b.n_elem);
        const int64_t e = r / d.n_tf % b.n_elem;
        const KT* c = ctab + (size_t)(e * d.na + a) * d.rec + f * d.P;
        const int JL = d.JL;
        const KT* ph = phi + ((size_t)i * d.G + j / JL) * d.phi_row + j % JL;
        KT s = 0;
        for (int p = 0; p < d.P; p++) s += c[p] * ph[p * JL];
        ke[b.group_base[a] + (e * d.n_tf + i) * b.ld + x] = s;
    }
    if (d.has_rhs) {
        int64_t u = t;
        for (int g = 0; g < b.n_rgroups; g++) {
            const int64_t n = (int64_t)b.rn_elem * b.rgroup_ntf[g];
            if (u < n) {
                const int64_t e = u / b.rgroup_ntf[g];
                const int k = b.rgroup_k[g] + (int)(u - e * b.rgroup_ntf[g]);
                ke[b.rgroup_base[g] + u] = (KT)-((double)rtab[d.rbase[k] + e * d.rstride] * d.rphi[k]);
                break;
            }
            u -= n;
        }
    }
}

hipError_t launch_direct_ke(const DirectDev& d, const DirectBuild& b, bool fp64, const void* ctab, const void* rtab, void* ke,
                            hipStream_t st) {
    int64_t n = (int64_t)d.na * b.n_elem * d.n_tf * d.nb * d.n_dof, nr = 0;
    if (d.has_rhs)
        for (int g = 0; g < b.n_rgroups; g++) nr += (int64_t)b.rn_elem * b.rgroup_ntf[g];
    n = std::max(n, nr);
    if (n == 0) return hipSuccess;
    const unsigned grid = (unsigned)((n + 255) / 256);
    if (fp64) hipLaunchKernelGGL((direct_ke_kernel<double>), dim3(grid), dim3(256), 0, st, d, b, (const double*)ctab, (const double*)rtab, (double*)ke);
    else hipLaunchKernelGGL((direct_ke_kernel<float>), dim3(grid), dim3(256), 0, st, d, b, (const float*)ctab, (const float*)rtab, (float*)ke);
    return hipGetLastError();
}

}  // namespace slx
