// The one-tile-per-element kernel (kernels/tile.h) compiled for one slice: its
// text follows a namespace tj with the slice's constants (coefjit.cpp).
//
// What bounds it: order-3 quadrangles (16 x 16, 25 points) the memory traffic
// of the coefficient table and Ke, 2.7 TB/s; larger tiles the matrix and vector
// ALUs in turn (two to four waves a SIMD).  The slice is known, so only its (tf,
// dof) derivative pairs are multiplied (D[pair][q], a lane's Gauss points in one
// read, instead of 4 x 4 matrices); the weighted dof table and the P fragments stay
// in registers for the whole launch where they fit (H_REG, P_REG), else in LDS; a
// wave loads the coefficients of EB elements at once and never waits for another
// wave; the operands are swapped (Ke^T = Q_e^T P), so that a lane holds consecutive
// entries of a row of Ke.  The arithmetic is tile.hip's: the same scaling, splits
// and products in the same order.  Measured, tile.hip -> here: 5.5e5 order-3
// quadrangles FP16 split 634 -> 313 us (EB = 1: 430); 1.6e4 order-3 prisms BF16 split,
// stiffness 222 -> 164 us, mass 158 -> 48 us; 48000 order-2 H(curl) tetrahedra in 24
// buckets 130 -> 82 us.
// N_STORE: the columns or, where no other slice shares the rows, with the padding
// up to ld (zeros).  Rows of whole lines are stored past the caches (quadrangles
// 320 us, else 342; H(curl) 82 us, else 92, and the reduction 165 us, else 205);
// others not, since their pieces of a line meet in L2 (mass matrices of prisms
// 48 us, else 67).
namespace slx {

typedef _Float16 tj_half2 __attribute__((ext_vector_type(2)));
typedef _Float16 tj_half8 __attribute__((ext_vector_type(8)));
typedef __bf16 tj_bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 tj_bf8 __attribute__((ext_vector_type(8)));
typedef float tj_f2 __attribute__((ext_vector_type(2)));
typedef float tj_f4 __attribute__((ext_vector_type(4)));
typedef float tj_f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned int tj_u4 __attribute__((ext_vector_type(4)));

namespace tj {
constexpr int QH = 8 / NA, NGPP = NKC * 4 * QH, NC = 16 * NTT, NPL = AR == 1 ? 3 : 2, HN = QH * NB;
constexpr int PASS = (NGPP + 63) / 64;
constexpr int P_WORDS = P_REG ? 0 : NKC * MTT * NPL * 64, H_FLOATS = H_REG ? 0 : NKC * NTT * 64 * HN;
constexpr int LDS = P_WORDS * 16 + H_FLOATS * 4 + WAVES * EB * NP * NGPP * 4;

// the eight values of a lane as the arithmetic's operand words
__device__ inline void split(const float (&v)[8], tj_u4 (&qp)[NPL]) {
    if constexpr (AR == 2) {
        qp[0] = __builtin_bit_cast(tj_u4, tj_f4{v[0], v[1], v[2], v[3]});
        qp[1] = __builtin_bit_cast(tj_u4, tj_f4{v[4], v[5], v[6], v[7]});
    } else if constexpr (AR == 1) {
#pragma unroll
        for (int x = 0; x < 4; x++) {
            tj_f2 r{v[2 * x], v[2 * x + 1]};
#pragma unroll
            for (int pl = 0; pl < NPL; pl++) {
                const tj_bf2 b = __builtin_convertvector(r, tj_bf2);
                qp[pl][x] = __builtin_bit_cast(unsigned int, b);
                r[0] -= (float)b[0];
                r[1] -= (float)b[1];
            }
        }
    } else {
        // v - hi and its rounding in one instruction (v_fma_mixlo/mixhi_f16; a
        // constant -1 would fold to a conversion and a subtraction)
        float neg = -1.f;
        asm("" : "+s"(neg));
#pragma unroll
        for (int x = 0; x < 4; x++) {
            const tj_half2 hi = __builtin_convertvector(tj_f2{v[2 * x], v[2 * x + 1]}, tj_half2);
            const tj_half2 lo{(_Float16)__builtin_fmaf((float)hi[0], neg, v[2 * x]), (_Float16)__builtin_fmaf((float)hi[1], neg, v[2 * x + 1])};
            qp[0][x] = __builtin_bit_cast(unsigned int, hi);
            qp[1][x] = __builtin_bit_cast(unsigned int, lo);
        }
    }
}

__device__ inline tj_f4 product(const tj_u4 p, const tj_u4 q, tj_f4 acc) {
    if constexpr (AR == 1) {
        const tj_bf8 a = __builtin_bit_cast(tj_bf8, p), b = __builtin_bit_cast(tj_bf8, q);
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, acc, 0, 0, 0);
    } else {
        const tj_half8 a = __builtin_bit_cast(tj_half8, p), b = __builtin_bit_cast(tj_half8, q);
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(b, a, acc, 0, 0, 0);
    }
}

// Maximum over the wave of values >= 0, on their bits (NaN counts as large).
__device__ inline float wave_max(float f) {
    int m = __builtin_bit_cast(int, f);
#define TJ_DPP(ctrl) m = max(m, __builtin_amdgcn_update_dpp(0, m, ctrl, 0xf, 0xf, true))
    TJ_DPP(0xB1);   // quad_perm 1 0 3 2
    TJ_DPP(0x4E);   // quad_perm 2 3 0 1
    TJ_DPP(0x141);  // row_half_mirror
    TJ_DPP(0x140);  // row_mirror
#undef TJ_DPP
    return __builtin_bit_cast(float, max(max(__builtin_amdgcn_readlane(m, 0), __builtin_amdgcn_readlane(m, 16)),
                                         max(__builtin_amdgcn_readlane(m, 32), __builtin_amdgcn_readlane(m, 48))));
}
}  // namespace tj

extern "C" __global__ void __launch_bounds__(64 * tj::WAVES, tj::OCC)
    slx_tile(TJ_ARG, const unsigned char* __restrict__ cbase, int qfast, float* __restrict__ ke) {
    using namespace tj;
    TJ_JOB;
    const int n_elem = (int)job.n_elem;
    __shared__ __attribute__((aligned(16))) unsigned char lds[LDS];
    tj_u4* Pl = reinterpret_cast<tj_u4*>(lds);
    float* Hl = reinterpret_cast<float*>(lds + P_WORDS * 16);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, jl = lane & 15;
    float* Dl = Hl + H_FLOATS + w * (EB * NP * NGPP);  // this wave's [element of the batch][pair][q]
    const SLX_GLOBAL tj_f4* tq4 = (const SLX_GLOBAL tj_f4*)job.t.tq;
    const SLX_GLOBAL tj_u4* af = (const SLX_GLOBAL tj_u4*)job.t.afrag;
    // entry k = point * NB + derivative of a lane's piece of the dof table
    auto h_entry = [&](int c, int jt, int ln, int k) {
        return tq4[((4 * c + (ln >> 4)) * QH + k / NB) * NC + jt * 16 + (ln & 15)][B_OF[k % NB]];
    };
    // pieces as float4 planes and, for the last two entries, a float2 plane
    auto h_at = [&](int c, int jt, int ln, int k) {
        return (c * NTT + jt) * 64 * HN + (k < HN / 4 * 4 ? k / 4 * 256 + ln * 4 + k % 4 : HN / 4 * 256 + ln * 2 + k % 4);
    };
    float hr[H_REG ? NKC : 1][H_REG ? NTT : 1][HN];
    tj_u4 pr[P_REG ? NKC : 1][P_REG ? MTT : 1][NPL];
    if constexpr (H_REG) {
#pragma unroll
        for (int c = 0; c < NKC; c++)
#pragma unroll
            for (int jt = 0; jt < NTT; jt++)
#pragma unroll
                for (int k = 0; k < HN; k++) hr[c][jt][k] = h_entry(c, jt, lane, k);
    } else {
        for (int x = tid; x < NKC * NTT * 64; x += 64 * WAVES)
#pragma unroll
            for (int k = 0; k < HN; k++) Hl[h_at(x / 64 / NTT, x / 64 % NTT, x & 63, k)] = h_entry(x / 64 / NTT, x / 64 % NTT, x & 63, k);
    }
    if constexpr (P_REG) {
#pragma unroll
        for (int c = 0; c < NKC; c++)
#pragma unroll
            for (int mt = 0; mt < MTT; mt++)
#pragma unroll
                for (int pl = 0; pl < NPL; pl++) pr[c][mt][pl] = af[((c * MTT + mt) * NPL + pl) * 64 + lane];
    } else {
        for (int x = tid; x < P_WORDS; x += 64 * WAVES) Pl[x] = af[x];
    }
    if constexpr (!P_REG || !H_REG) __syncthreads();
    // EB elements per wave at a time: the coefficients are [slot][point][element]
    // (a lane takes EB consecutive elements of its point in one load) or, with
    // qfast, [slot][element][point].  Workgroup w runs on XCD w % 8 (the grid is a
    // multiple of 8): each XCD takes a contiguous eighth of the elements and its
    // workgroups neighbouring batches, so that the pieces of the table's NT * NGP
    // rows that are read together are neighbours too.
    constexpr int step = EB * WAVES;
    const int n_batch = (n_elem + step - 1) / step, xcd = blockIdx.x % 8;
    const int e_end = (int)min((int64_t)n_elem, (int64_t)n_batch * (xcd + 1) / 8 * step);
    const int64_t e_step = (int64_t)(gridDim.x / 8) * step;
    const float* ctab = reinterpret_cast<const float*>(cbase + job.coff);
    const int64_t stride = (int64_t)NGP * n_elem, es = qfast ? NGP : 1, ps = qfast ? 1 : (int64_t)n_elem;
    float cv[PASS][NT][EB];
    auto load_c = [&](int64_t e) {
#pragma unroll
        for (int p = 0; p < PASS; p++) {
            const int q = lane + 64 * p;
            const float* cq = ctab + e * es + (int64_t)q * ps;
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int x = 0; x < EB; x++) cv[p][t][x] = 0.f;
            if (q < NGP) {
                if (EB == 4 && !qfast && e + EB <= e_end) {
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        const tj_f4u v = *reinterpret_cast<const tj_f4u*>(cq + TERM_SLOT[t] * stride);
#pragma unroll
                        for (int x = 0; x < EB; x++) cv[p][t][x] = v[x];
                    }
                } else {
#pragma unroll
                    for (int x = 0; x < EB; x++)
                        if (e + x < e_end)
#pragma unroll
                            for (int t = 0; t < NT; t++) cv[p][t][x] = cq[TERM_SLOT[t] * stride + x * es];
                }
            }
        }
    };
    const float tqmax = job.t.tqmax, a_unscale = job.t.a_unscale;
    const int64_t ld = job.t.ke_ld;
    float* const ke0 = ke + job.t.ke_base;
    int64_t eb = ((int64_t)n_batch * xcd / 8 + blockIdx.x / 8) * step + EB * w;
    for (; eb < e_end; eb += e_step) {
        load_c(eb);
        // coefficient of every derivative pair at the lane's Gauss points
        float s[PASS][NP][EB], m[EB], unscs[EB];
#pragma unroll
        for (int x = 0; x < EB; x++) {
            m[x] = 0.f;
#pragma unroll
            for (int p = 0; p < PASS; p++) {
#pragma unroll
                for (int y = 0; y < NP; y++) s[p][y][x] = 0.f;
#pragma unroll
                for (int t = 0; t < NT; t++) s[p][TERM_PAIR[t]][x] += cv[p][t][x];
#pragma unroll
                for (int a = 0; a < NA; a++) {
                    float r = 0.f;
#pragma unroll
                    for (int y = 0; y < NP; y++)
                        if (PAIR_A[y] == a) r += fabsf(s[p][y][x]);
                    m[x] = __builtin_bit_cast(int, r) > __builtin_bit_cast(int, m[x]) ? r : m[x];
                }
            }
        }
#pragma unroll
        for (int x = 0; x < EB; x++) {
            // power-of-two scale: |Q| <= max_q,a sum_b |D| * max |tq|  ->  [128, 256)
            const float bound = wave_max(m[x]) * tqmax;
            const int bits = __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, bound)), ef = bits >> 23;  // uniform
            int ex = 8;  // zero, subnormal or not finite: unscaled
            float sc = 1.f;
            if (ef >= 8 && ef < 255) {
                ex = ef - 126;  // bound in [2^(ex - 1), 2^ex)
                sc = __builtin_bit_cast(float, (261 - ef) << 23);  // 2^(8 - ex)
            }
            unscs[x] = ldexpf(a_unscale, ex - 8);
#pragma unroll
            for (int p = 0; p < PASS; p++)
                if (64 * (p + 1) <= NGPP || lane + 64 * p < NGPP)
#pragma unroll
                    for (int y = 0; y < NP; y++) Dl[(x * NP + y) * NGPP + lane + 64 * p] = sc * s[p][y][x];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (int x = 0; x < EB; x++) {
            const int64_t e = eb + x;
            if (e >= e_end) break;
            float unsc = unscs[0];
#pragma unroll
            for (int y = 1; y < EB; y++)
                if (y == x) unsc = unscs[y];
            const float* dl = Dl + x * (NP * NGPP) + g * QH;
            tj_f4 acc[MTT][NTT];
#pragma unroll
            for (int mt = 0; mt < MTT; mt++)
#pragma unroll
                for (int jt = 0; jt < NTT; jt++) acc[mt][jt] = tj_f4{0.f, 0.f, 0.f, 0.f};
            auto chunk = [&](int c) {
                float d[NP][QH];
#pragma unroll
                for (int x = 0; x < NP; x++) {
                    const float* dx = dl + x * NGPP + 4 * QH * c;
                    if constexpr (QH == 2) {
                        const tj_f2 v = *reinterpret_cast<const tj_f2*>(dx);
                        d[x][0] = v[0];
                        d[x][1] = v[1];
                    } else {
#pragma unroll
                        for (int y = 0; y < QH / 4; y++) {
                            const tj_f4 v = *reinterpret_cast<const tj_f4*>(dx + 4 * y);
#pragma unroll
                            for (int z = 0; z < 4; z++) d[x][4 * y + z] = v[z];
                        }
                    }
                }
                tj_u4 pp[MTT][NPL];
#pragma unroll
                for (int mt = 0; mt < MTT; mt++)
#pragma unroll
                    for (int pl = 0; pl < NPL; pl++) {
                        if constexpr (P_REG) pp[mt][pl] = pr[c][mt][pl];
                        else pp[mt][pl] = Pl[((c * MTT + mt) * NPL + pl) * 64 + lane];
                    }
#pragma unroll
                for (int jt = 0; jt < NTT; jt++) {
                    float h[HN];
                    if constexpr (H_REG) {
#pragma unroll
                        for (int k = 0; k < HN; k++) h[k] = hr[c][jt][k];
                    } else {
                        const float* hp = Hl + (c * NTT + jt) * 64 * HN;
#pragma unroll
                        for (int y = 0; y < HN / 4; y++) {
                            const tj_f4 v = *reinterpret_cast<const tj_f4*>(hp + y * 256 + lane * 4);
#pragma unroll
                            for (int z = 0; z < 4; z++) h[4 * y + z] = v[z];
                        }
                        if constexpr (HN % 4 != 0) {
                            const tj_f2 v = *reinterpret_cast<const tj_f2*>(hp + HN / 4 * 256 + lane * 2);
                            h[HN / 4 * 4] = v[0];
                            h[HN / 4 * 4 + 1] = v[1];
                        }
                    }
                    // the lane's eight Q_e entries of the column tile
                    float v[8];
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        v[k] = 0.f;
                        if (k / NA < QH)
#pragma unroll
                            for (int x = 0; x < NP; x++)
                                if (PAIR_A[x] == k % NA) v[k] += d[x][k / NA] * h[k / NA * NB + PAIR_B[x]];
                    }
                    tj_u4 qp[NPL];
                    split(v, qp);
                    if constexpr (AR == 2) {
#pragma unroll
                        for (int k = 0; k < 8; k++)
#pragma unroll
                            for (int mt = 0; mt < MTT; mt++) {
                                const float x = __builtin_bit_cast(tj_f4, pp[mt][k >> 2])[k & 3];
                                acc[mt][jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[k], x, acc[mt][jt], 0, 0, 0);
                            }
                    } else {
                        // FP16: hi hi, hi lo, lo hi; BF16: hi hi, hi mid, mid hi, hi lo, mid mid, lo hi
                        constexpr int PP[6] = {0, 0, 1, 0, 1, 2}, QQ[6] = {0, 1, 0, 2, 1, 0};
#pragma unroll
                        for (int x = 0; x < (AR == 1 ? 6 : 3); x++)
#pragma unroll
                            for (int mt = 0; mt < MTT; mt++) acc[mt][jt] = product(pp[mt][PP[x]], qp[QQ[x]], acc[mt][jt]);
                    }
                }
            };
            if constexpr (H_REG || P_REG) {
#pragma unroll
                for (int c = 0; c < NKC; c++) chunk(c);
            } else {
#pragma unroll 1
                for (int c = 0; c < NKC; c++) chunk(c);
            }
            float* out = ke0 + e * N_TF * ld;
#pragma unroll
            for (int jt = 0; jt < NTT; jt++)
#pragma unroll
                for (int mt = 0; mt < MTT; mt++) {
                    const tj_f4 v = acc[mt][jt] * unsc;
                    const int i = mt * 16 + jl, j = jt * 16 + 4 * g;
                    float* o = out + i * ld + j;
                    if (i < N_TF) {
                        if (j + 4 <= N_STORE) {
                            if constexpr (N_STORE % 16 == 0) __builtin_nontemporal_store(v, reinterpret_cast<tj_f4u*>(o));
                            else *reinterpret_cast<tj_f4u*>(o) = v;
                        } else {
#pragma unroll
                            for (int r = 0; r < 4; r++)
                                if (j + r < N_STORE) o[r] = v[r];
                        }
                    }
                }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the coefficients are read before the next elements' are written
        __builtin_amdgcn_wave_barrier();
    }
}
}  // namespace slx
