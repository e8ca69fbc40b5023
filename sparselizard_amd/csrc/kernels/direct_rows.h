// Kernel and launchers of the row-wise assembly (direct.hip); instantiated for
// FP32 and FP64 values in direct_f32.hip and direct_f64.hip.
#pragma once
#include <algorithm>
#include <utility>
#include "direct.h"

namespace slx {

typedef float dfloat4 __attribute__((ext_vector_type(4)));
typedef double ddouble2 __attribute__((ext_vector_type(2)));
typedef uint64_t du64x2 __attribute__((ext_vector_type(2)));

template <typename KT>
struct DirectVec;
template <>
struct DirectVec<float> {
    typedef dfloat4 type;
    static constexpr int N = 4;
};
template <>
struct DirectVec<double> {
    typedef ddouble2 type;
    static constexpr int N = 2;
};

// N entries (a multiple of 4) from 16-byte aligned memory
template <typename KT, int N>
__device__ inline void direct_load(const KT* p, KT (&v)[N]) {
    typedef typename DirectVec<KT>::type V;
    constexpr int W = DirectVec<KT>::N;
#pragma unroll
    for (int k = 0; k < N; k += W) {
        const V x = *reinterpret_cast<const V*>(p + k);
#pragma unroll
        for (int c = 0; c < W; c++) v[k + c] = x[c];
    }
}

// The right-hand side of one free row: its entries in accumulation order
// (rawvec.cpp:216-254), four loads in flight.  The products are FP64 in every
// mode: with FP32 ones the rounded Gauss-point sums, the same in all entries, made
// the sums of FP32 coefficients 1.3 times as far off as a sum over the Gauss points.
template <typename KT>
__device__ inline void direct_rhs_row(const DirectDev& d, const KT* __restrict__ rtab, const double* __restrict__ rphi, int64_t r,
                                      double* __restrict__ rhs) {
    const uint32_t kmask = (1u << d.rib) - 1u;
    double s = 0.0;
    int64_t k = d.rptr[r];
    const int64_t k1 = d.rptr[r + 1];
    for (; k < k1; k += 4) {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t w = k + u < k1 ? d.rseg[k + u] : 0u;
            const uint32_t f = w & kmask;
            v[u] = k + u < k1 ? -((double)rtab[d.rbase[f] + (int64_t)(w >> d.rib) * d.rstride] * rphi[f]) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) s += v[u];
    }
    rhs[d.free_dofs[r]] = s;
}

__device__ inline uint64_t direct_lane64(uint64_t v, int lane) {
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, lane), hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), lane);
    return (uint64_t)hi << 32 | lo;
}

// One row of a wave's batch: its A and D positions, first segment, slot block.
struct DirectRow {
    uint64_t a, d;
    int64_t k0, sb;
    int nk;
};

// The value of lane O of the G lanes that share a row (G = 1, 2 or 4: lanes of
// one quad).
template <int G, int O>
__device__ inline uint32_t direct_bcast32(uint32_t v) {
    constexpr int perm = G == 4 ? 0x55 * O : (O | O << 2 | (O + 2) << 4 | (O + 2) << 6);
    return G == 1 ? v : (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, perm, 0xf, 0xf, true);
}
template <int G, int O>
__device__ inline float direct_bcast(float v) {
    return __uint_as_float(direct_bcast32<G, O>(__float_as_uint(v)));
}
template <int G, int O>
__device__ inline double direct_bcast(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint64_t lo = direct_bcast32<G, O>((uint32_t)u), hi = direct_bcast32<G, O>((uint32_t)(u >> 32));
    return __longlong_as_double((long long)(hi << 32 | lo));
}

// Coefficient K of a segment whose 16-byte pieces the row's lanes hold in turn.
template <typename KT, int G, int N, int K>
__device__ inline KT direct_coef(const KT (&c)[N]) {
    constexpr int W = DirectVec<KT>::N, piece = K / W;
    return direct_bcast<G, piece % G>(c[piece / G * W + K % W]);
}

template <typename KT, int G, int N, int K0, int P, int... I>
__device__ inline void direct_coefs(const KT (&c)[N], KT (&out)[P], std::integer_sequence<int, I...>) {
    ((out[I] = direct_coef<KT, G, N, K0 + I>(c)), ...);
}

// t[b][jj] = sum_p C[b][p] phi[p][jj] of one dof field after the other.
template <typename KT, int G, int N, int P, int JL, int PJ, int B>
__device__ inline void direct_field(const KT (&c)[N], const KT (&ph)[PJ], KT* t) {
    KT v[P];
    direct_coefs<KT, G, N, B * P, P>(c, v, std::make_integer_sequence<int, P>());
#pragma unroll
    for (int jj = 0; jj < JL; jj++) {
        KT s = 0;
#pragma unroll
        for (int p = 0; p < P; p++) s += v[p] * ph[p * JL + jj];
        t[B * JL + jj] = s;
    }
}
template <typename KT, int G, int N, int NB, int P, int JL, int PJ, int... B>
__device__ inline void direct_sums(const KT (&c)[N], const KT (&ph)[PJ], KT (&t)[NB * JL], std::integer_sequence<int, B...>) {
    (direct_field<KT, G, N, P, JL, PJ, B>(c, ph, t), ...);
}

// Waves per SIMD the registers are limited to.
template <typename KT, int NB, int P>
constexpr int direct_waves() {
    return NB * P * (int)sizeof(KT) <= 16 ? 4 : sizeof(KT) == 4 ? 3 : 2;
}

// Blocks below mat_blocks stay for the launch; their waves walk batches of
// rpw rows (an LDS accumulator of acc_stride doubles each).  The blocks above
// take one right-hand-side row per lane.
//
// A row has few segments (6 on an edge, 24 at a vertex of a tetrahedral mesh)
// and each costs a chain of dependent loads: descriptor, segment word,
// coefficients.  The waves therefore run ahead: NBUF segments' coefficients
// are in flight per row, the last ones of a batch being the first of the
// next, whose descriptors and segment words were loaded during the batch.
// Loads past a row's end read the first words behind it (the arrays are padded)
// and are not summed.
//
// The G lanes of a row load its coefficients once, 16 bytes each in turn, and
// hand them around inside the multiply-adds (quad permutes).  Loading all of
// them in every lane instead kept the address unit busy 80 % of the time and
// bound the kernel (64 lanes x 16 bytes of 12 records: 45 cycles an
// instruction, seven per segment).
//
// Measured at 48^3 x 6 P2 elasticity tetrahedra (6e8 element-matrix entries,
// 2.3e8 nonzeros): 0.65 ms for the 2.3e6 edge rows (12 waves on a CU; vector
// ALU and LDS each about half busy, 2.0 GB moved), 0.39 ms for the 3.4e5 vertex
// rows (6 waves: their accumulators fill the LDS), against 0.78 ms of the
// element kernel and 1.16 ms of the reduction.
template <typename KT, typename ST, int NB, int P, int JL, int G>
__global__ void __launch_bounds__((256 * direct_waves<KT, NB, P>()), (direct_waves<KT, NB, P>())) direct_rows(DirectDev d, const KT* __restrict__ ctab, const KT* __restrict__ rtab, int64_t pos0,
                                                   int64_t pos1, unsigned mat_blocks, int rpw, int acc_stride, int write_lanes,
                                                   double* __restrict__ Aval, double* __restrict__ Dval, double* __restrict__ rhs) {
    constexpr int EN = NB * JL;                               // entries per lane and segment
    constexpr int SW = (EN * (int)sizeof(ST) + 3) / 4;        // their slots, in 32-bit words
    constexpr int W = DirectVec<KT>::N;                       // values per 16 bytes
    constexpr int PIECES = (NB * P + W - 1) / W;              // of a segment's coefficients
    constexpr int LP = (PIECES + G - 1) / G, KC = LP * W;     // a lane's pieces and values
    constexpr int PJ = (P * JL + 3) / 4 * 4;                  // table entries per lane
    constexpr int NBUF = NB * P * (int)sizeof(KT) <= 48 ? 4 : sizeof(KT) == 4 ? 3 : 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char direct_lds[];
    const KT* phi_g;
    if constexpr (sizeof(KT) == 4) phi_g = (const KT*)d.phi32;
    else phi_g = (const KT*)d.phi64;
    if (blockIdx.x >= mat_blocks) {
        const int64_t r = (int64_t)(blockIdx.x - mat_blocks) * blockDim.x + threadIdx.x;
        if (r < d.nrows) direct_rhs_row<KT>(d, rtab, d.rphi, r, rhs);
        return;
    }
    const int nphi = d.n_tf * G * PJ;
    KT* phi = reinterpret_cast<KT*>(direct_lds);
    double* acc_all = reinterpret_cast<double*>(direct_lds + ((size_t)nphi * sizeof(KT) + 15) / 16 * 16);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    double* accw = acc_all + (size_t)wave * rpw * acc_stride;
    for (int x = threadIdx.x; x < nphi; x += blockDim.x) phi[x] = phi_g[x];
    for (int x = lane; x < rpw * acc_stride; x += 64) accw[x] = 0.0;
    __syncthreads();
    // workgroup w runs on XCD w % 8: each XCD takes one contiguous eighth of
    // the batches, its waves neighbouring ones at a time
    const int64_t nbatch = (pos1 - pos0 + rpw - 1) / rpw;
    const int xcd = blockIdx.x % 8;
    const int64_t b_end = nbatch * (xcd + 1) / 8, b_step = (int64_t)(mat_blocks / 8) * waves;
    int64_t batch = nbatch * xcd / 8 + (int64_t)(blockIdx.x / 8) * waves + wave;
    if (batch >= b_end) return;
    const int row = lane / G, l = lane % G;
    const uint64_t M48 = 0xFFFFFFFFFFFFull;
    auto load_row = [&](int64_t bt) {
        DirectRow r{0, 0, 0, 0, 0};
        const int64_t pos = pos0 + bt * rpw + row;
        if (bt < b_end && row < rpw && pos < pos1) {
            const du64x2 w01 = *reinterpret_cast<const du64x2*>(d.desc + 4 * pos);
            const du64x2 w23 = *reinterpret_cast<const du64x2*>(d.desc + 4 * pos + 2);
            r.a = w01[0];
            r.d = w01[1];
            r.k0 = (int64_t)(w23[0] & M48);
            r.nk = (int)(w23[0] >> 48);
            r.sb = (int64_t)w23[1];
        }
        return r;
    };
    double* acc = accw + (size_t)min(row, rpw - 1) * acc_stride;
    const uint32_t imask = (1u << d.ib) - 1u;
    const int n_dof = d.n_dof;
    auto load_words = [&](const DirectRow& r, int k, uint32_t (&w)[NBUF]) {
#pragma unroll
        for (int u = 0; u < NBUF; u++) w[u] = d.seg[r.k0 + min(k, r.nk) + u];
    };
    auto load_seg = [&](const DirectRow& r, int k, uint32_t w, KT (&c)[KC], uint32_t (&sl)[SW]) {
        const KT* rec = ctab + (size_t)(w >> d.ib) * (size_t)d.rec;
#pragma unroll
        for (int x = 0; x < LP; x++) {
            const int piece = min(x * G + l, PIECES - 1);
            const typename DirectVec<KT>::type v = *reinterpret_cast<const typename DirectVec<KT>::type*>(rec + piece * W);
#pragma unroll
            for (int z = 0; z < W; z++) c[x * W + z] = v[z];
        }
        const uint32_t* sp = d.slots + ((size_t)(r.sb + min(k, r.nk)) * G + l) * SW;
#pragma unroll
        for (int u = 0; u < SW; u++) sl[u] = sp[u];
    };
    DirectRow cur = load_row(batch), nxt = load_row(batch + b_step);
    uint32_t w[NBUF], wn[NBUF];
    KT c[NBUF][KC];
    uint32_t sl[NBUF][SW];
    load_words(cur, 0, w);
    load_words(cur, NBUF, wn);
#pragma unroll
    for (int u = 0; u < NBUF; u++) load_seg(cur, u, w[u], c[u], sl[u]);
    while (true) {
        uint32_t x0[NBUF], x1[NBUF];  // the next batch's first words
        load_words(nxt, 0, x0);
        load_words(nxt, NBUF, x1);
        const DirectRow nxt2 = load_row(batch + 2 * b_step);
        for (int kb = 0;; kb += NBUF) {
            const bool more = __any(kb + NBUF < cur.nk);
            uint32_t wf[NBUF];
            if (more) load_words(cur, kb + 2 * NBUF, wf);
#pragma unroll
            for (int u = 0; u < NBUF; u++) {
                if (kb + u < cur.nk) {
                    KT ph[PJ];
                    direct_load<KT, PJ>(phi + ((int)(w[u] & imask) * G + l) * PJ, ph);
                    KT t[EN];
                    direct_sums<KT, G, KC, NB, P, JL, PJ>(c[u], ph, t, std::make_integer_sequence<int, NB>());
#pragma unroll
                    for (int jj = 0; jj < JL; jj++)
                        if (l * JL + jj < n_dof)
#pragma unroll
                            for (int b = 0; b < NB; b++) {
                                const int x = b * JL + jj;
                                const uint32_t slot = sizeof(ST) == 1 ? (sl[u][x / 4] >> (8 * (x % 4))) & 0xFFu
                                                                      : (sl[u][x / 2] >> (16 * (x % 2))) & 0xFFFFu;
                                // LDS FP64 add without return; one wave's LDS operations complete in
                                // issue order, so the order of the additions is the program's
                                (void)atomicAdd(&acc[slot], (double)t[x]);
                            }
                }
                if (more) load_seg(cur, kb + NBUF + u, wn[u], c[u], sl[u]);
                else load_seg(nxt, u, x0[u], c[u], sl[u]);
            }
            if (!more) break;
#pragma unroll
            for (int u = 0; u < NBUF; u++) {
                w[u] = wn[u];
                wn[u] = wf[u];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // the wave writes its rows (A then D entries, both in the row's
        // accumulator) and clears them for the next batch
        auto put = [&](uint64_t a, uint64_t dd, int x, double v) {
            const int lenA = (int)(a >> 48), len = lenA + (int)(dd >> 48);
            double* p = x < lenA ? Aval + (int64_t)(a & M48) : Dval + (int64_t)(dd & M48) - lenA;
            if (x < len) p[x] = v;
        };
        if (write_lanes == 64) {
            // two rows' first 128 entries in flight together
            for (int r0 = 0; r0 < rpw; r0 += 2) {
                double v[2][2];
#pragma unroll
                for (int y = 0; y < 2; y++)
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        double* p = accw + (size_t)min(r0 + y, rpw - 1) * acc_stride + min(lane + 64 * h, acc_stride - 1);
                        v[y][h] = *p;
                    }
#pragma unroll
                for (int y = 0; y < 2; y++) {
                    if (r0 + y >= rpw) break;
                    const uint64_t a = direct_lane64(cur.a, (r0 + y) * G), dd = direct_lane64(cur.d, (r0 + y) * G);
                    double* ar = accw + (size_t)(r0 + y) * acc_stride;
                    const int len = (int)(a >> 48) + (int)(dd >> 48);
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        put(a, dd, lane + 64 * h, v[y][h]);
                        if (lane + 64 * h < acc_stride) ar[lane + 64 * h] = 0.0;
                    }
                    for (int x = lane + 128; x < len; x += 64) {
                        put(a, dd, x, ar[x]);
                        ar[x] = 0.0;
                    }
                }
            }
        } else {
            // short rows: write_lanes lanes each
            const int wr = lane / write_lanes, wl = lane - wr * write_lanes, rstep = 64 / write_lanes;
            for (int r0 = 0; r0 < rpw; r0 += rstep) {
                const int rr = r0 + wr;
                const int src = min(rr, rpw - 1) * G;
                const uint64_t a = __shfl(cur.a, src, 64), dd = __shfl(cur.d, src, 64);
                if (rr < rpw && wl < acc_stride) {
                    double* ar = accw + (size_t)rr * acc_stride;
                    put(a, dd, wl, ar[wl]);
                    ar[wl] = 0.0;
                }
            }
        }
        batch += b_step;
        if (batch >= b_end) break;
        // the rows' spare entries, which took the absent columns and may be a column
        // of the next row there: all rows at once (a store a row cost 0.9 % at 48^3)
        acc[(int)(cur.a >> 48) + (int)(cur.d >> 48)] = 0.0;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        cur = nxt;
        nxt = nxt2;
#pragma unroll
        for (int u = 0; u < NBUF; u++) {
            w[u] = x0[u];
            wn[u] = x1[u];
        }
    }
}

template <typename KT, typename ST, int NB, int P, int JL, int G>
static hipError_t launch_direct_t(const DirectDev& d, const DirectLaunch& q) {
    const size_t phi = direct_phi_bytes(d, sizeof(KT) == 8);
    const int stride = direct_stride(q.len);
    // the workgroup size that puts the most waves on a CU: several of up to four
    // waves that leave a tenth of the LDS free, or one larger (three of 53 KB
    // did not start together: the third ran behind the other two, edge rows
    // 0.89 ms; one of twelve waves: 0.65 ms)
    constexpr int cap = 4 * direct_waves<KT, NB, P>();
    int waves = 0, rpw = 64 / G, best = 0;
    for (int t = 0; t < cap; t++) {
        const int w = t < 4 ? 4 - t : t + 1;
        const size_t need = phi + (size_t)w * rpw * stride * 8;
        if (need > SLX_DIRECT_LDS) continue;
        const int blocks = (int)std::min<size_t>(cap / w, std::max<size_t>(1, SLX_DIRECT_CU_LDS / need));
        if (w * blocks > best) {
            best = w * blocks;
            waves = w;
        }
    }
    if (waves == 0) {
        // rows too long for a full wave of them
        waves = 1;
        while (rpw > 1 && phi + (size_t)rpw * stride * 8 > SLX_DIRECT_LDS) rpw--;
        best = 1;
    }
    const size_t lds = phi + (size_t)waves * rpw * stride * 8;
    if (lds > SLX_DIRECT_LDS) return hipErrorInvalidValue;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)direct_rows<KT, ST, NB, P, JL, G>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    // lanes that write a row: the row in one step, or the whole wave
    const int wlanes = q.len <= 8 ? 8 : q.len <= 16 ? 16 : q.len <= 32 ? 32 : 64;
    const int64_t rows = q.pos1 - q.pos0, rpb = (int64_t)waves * rpw;
    const int64_t fit = (int64_t)d.n_cu * std::max(1, best / waves);
    const unsigned mat = (unsigned)((std::min((rows + rpb - 1) / rpb, fit) + 7) / 8 * 8);
    const unsigned extra = q.with_rhs ? (unsigned)((d.nrows + waves * 64 - 1) / (waves * 64)) : 0u;
    hipLaunchKernelGGL((direct_rows<KT, ST, NB, P, JL, G>), dim3(mat + extra), dim3(waves * 64), lds, q.st, d, (const KT*)q.ctab,
                       (const KT*)q.rtab, q.pos0, q.pos1, mat, rpw, stride, wlanes, q.Aval, q.Dval, q.rhs);
    return hipGetLastError();
}

// (JL, G) of direct_shape; 16-bit slots (rows of 255 columns or more) only with four lanes
template <typename KT, int NB, int P>
static hipError_t launch_direct_j(const DirectDev& d, const DirectLaunch& q) {
    if (d.slot_bytes == 2) {
        if (d.G != 4) return hipErrorInvalidValue;
        if (d.JL <= 3) return launch_direct_t<KT, uint16_t, NB, P, 3, 4>(d, q);
        return launch_direct_t<KT, uint16_t, NB, P, 5, 4>(d, q);
    }
    if (d.G == 1) return launch_direct_t<KT, uint8_t, NB, P, 3, 1>(d, q);
    if (d.G == 2) return d.JL == 2 ? launch_direct_t<KT, uint8_t, NB, P, 2, 2>(d, q) : launch_direct_t<KT, uint8_t, NB, P, 3, 2>(d, q);
    if (d.JL == 3) return launch_direct_t<KT, uint8_t, NB, P, 3, 4>(d, q);
    return launch_direct_t<KT, uint8_t, NB, P, 5, 4>(d, q);
}

template <typename KT>
static hipError_t launch_direct_k(const DirectDev& d, const DirectLaunch& q) {
    if (d.nb == 1) return d.P == 4 ? launch_direct_j<KT, 1, 4>(d, q) : d.P == 9 ? launch_direct_j<KT, 1, 9>(d, q) : launch_direct_j<KT, 1, 12>(d, q);
    if (d.nb == 2) return d.P == 4 ? launch_direct_j<KT, 2, 4>(d, q) : launch_direct_j<KT, 2, 9>(d, q);
    return d.P == 9 ? launch_direct_j<KT, 3, 9>(d, q) : launch_direct_j<KT, 3, 12>(d, q);
}

}  // namespace slx
