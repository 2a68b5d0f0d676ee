// emtf_eval.h -- the objectives on MFMA accumulators and their derivatives (gfx950), shared by
// the epoch, polish (island.hip) and operator (objective.hip) kernels.
#pragma once
#include <hip/hip_runtime.h>
#include "emtf_math.h"
#include "emtf_types.h"

namespace emtf {

typedef float f16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float4 lds4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float f4(const float4& v, int e) { return e == 0 ? v.x : (e == 1 ? v.y : (e == 2 ? v.z : v.w)); }

// ---------------------------------------------------------------------------
// Objective of the lane's individual from its MFMA accumulators.
// Lane (col, h) holds z_j for j = 32 jt + 8 (r >> 2) + 4 h + (r & 3); the two
// halves accumulate the even / odd blocks of four rows in increasing j and
// are combined once.
// ZPAD: the caller's Q rows past D are zero, so z_j = +0 there; the objectives whose
// term at z = +0 is +0 (whose sums it leaves as they are, bit for bit: they start at
// +0 and never reach -0) and costs what any other row's does then add those rows
// unmasked.  (Weierstrass keeps the mask: at z = 0 its term takes the small-|z| branch,
// which would diverge from the other rows of the same slot.)
// ---------------------------------------------------------------------------
template <int FUNC>
constexpr bool zero_term_at_zero() {
    return FUNC == F_SPHERE || FUNC == F_ELLIPTIC || FUNC == F_ACKLEY || FUNC == F_RASTRIGIN ||
           FUNC == F_GRIEWANK || FUNC == F_SCHWEFEL || FUNC == F_REF_RASTRIGIN;
}

// The objective's terms and final combination in split form, for the polish's line search
// and the wide kernel's row tiles on several waves (terms of a row tile computed apart from
// the running sums): the same operations, in the same order, as objective() below, which
// keeps them inline for the epoch kernels' code.
//
// Rosenbrock's term of row j (z = z_j, zn = z_{j+1}); it counts when row j + 1 exists.
__device__ __forceinline__ float rosen_val(float z, float zn) {
    const float zz = z * z;
    const float a = zz - zn;
    const float b = z - 1.0f;
    float t1 = 100.0f * a;
    t1 = t1 * a;
    const float b2 = b * b;
    return t1 + b2;
}

// The term values of row j of every objective but Rosenbrock and (textbook) Weierstrass (v2:
// Ackley's cosine term, Griewank's 2 sin^2 or the reference's factor); the Weierstrass terms
// only for rows j < Dm (0 otherwise).
template <int FUNC>
__device__ __forceinline__ void row_vals(float z, int j, int Dm, const float* tab, float& v1, float& v2) {
    if constexpr (FUNC == F_SPHERE) {
        v1 = z * z;
    } else if constexpr (FUNC == F_ELLIPTIC) {
        const float zz = z * z;
        v1 = tab[j] * zz;
    } else if constexpr (FUNC == F_ACKLEY) {
        v1 = z * z;
        v2 = sinpi_sq(z);
    } else if constexpr (FUNC == F_RASTRIGIN) {
        const float zz = z * z;
        const float s20 = 20.0f * sinpi_sq(z);
        v1 = zz + s20;
    } else if constexpr (FUNC == F_GRIEWANK) {
        v1 = z * z;
        v2 = 2.0f * sinpi_sq(z * tab[j]);
    } else if constexpr (FUNC == F_WEIERSTRASS) {
        v1 = 0.0f;
        if (j < Dm) v1 = weier_term(z);
    } else if constexpr (FUNC == F_SCHWEFEL) {
        const float sq = sqrtf(__builtin_fabsf(z));
        const float tv = sq * 0.159154937f;
        v1 = z * sin2pi(tv);
    } else if constexpr (FUNC == F_REF_ACKLEY) {
        v1 = z * z;
        const float tz = 2.0f * z;
        v2 = cospi_f(tz);
    } else if constexpr (FUNC == F_REF_RASTRIGIN) {
        const float zz = z * z;
        const float tz = 2.0f * z;
        const float c = cospi_f(tz);
        const float t = 10.0f * c;
        const float v = zz - t;
        v1 = v + 10.0f;
    } else if constexpr (FUNC == F_REF_GRIEWANK) {
        v1 = z * z;
        const float q = z / tab[j];
        const float tq = q * 0.159154937f;
        const float t = 2.0f * sinpi_sq(tq);
        v2 = 1.0f - t;
    } else if constexpr (FUNC == F_REF_WEIERSTRASS) {
        v1 = 0.0f;
        if (j < Dm) v1 = weier_ref_term(z);
    }
}

// The running sums' start (s2: the reference Griewank's product).
template <int FUNC>
__device__ __forceinline__ void sums_start(float& s1, float& s2) {
    s1 = 0.0f;
    s2 = (FUNC == F_REF_GRIEWANK) ? 1.0f : 0.0f;
}

// Adds one row's term values into the lane's sums (s2: Ackley's cosine sum, Griewank's
// running 1 - prod cos) when the row counts.
template <int FUNC>
__device__ __forceinline__ void row_sum(float v1, float v2, bool in, float& s1, float& s2) {
    if (!in) return;
    s1 = s1 + v1;
    if constexpr (FUNC == F_ACKLEY || FUNC == F_REF_ACKLEY) {
        s2 = s2 + v2;
    } else if constexpr (FUNC == F_REF_GRIEWANK) {
        s2 = s2 * v2;
    } else if constexpr (FUNC == F_GRIEWANK) {
        const float om = 1.0f - s2;
        const float aq = v2 * om;
        s2 = s2 + aq;
    }
}

// The fitness from the two halves' sums (lane h holds its half's s1, s2; the other
// half's come over the cross-half shuffle).
template <int FUNC>
__device__ __forceinline__ float objective_tail(float s1, float s2, int D, const float* tab, int h) {
    const float o1 = __shfl_xor(s1, 32);
    const float S = s1 + o1;  // A + B (commutative)
    const float Df = (float)D;
    if constexpr (FUNC == F_ACKLEY) {
        const float o2 = __shfl_xor(s2, 32);
        const float C = s2 + o2;
        const float q = S / Df;
        const float r = sqrtf(q);
        const float a = -0.2f * r;
        const float t1 = -20.0f * expm1_f(a);
        const float c2 = C / Df;
        const float b = -2.0f * c2;
        const float t2 = 2.71828175f * expm1_f(b);
        return t1 - t2;
    } else if constexpr (FUNC == F_GRIEWANK) {
        const float o2 = __shfl_xor(s2, 32);
        const float qA = h ? o2 : s2;
        const float qB = h ? s2 : o2;
        const float om = 1.0f - qA;
        const float tq = qB * om;
        const float Qv = qA + tq;
        const float s4 = S / 4000.0f;
        return s4 + Qv;
    } else if constexpr (FUNC == F_SCHWEFEL) {
        // the constant from the task table: 418.982887 (textbook) or 418.9829 (reference)
        const float cd = tab[0] * Df;
        return cd - S;
    } else if constexpr (FUNC == F_REF_ACKLEY) {
        // -20 expf(-0.2 sqrtf(S / D)) - expf(C / D) + 20 + E with the reference's double
        // literals -0.2 and E = 2.718282 (SG-EMTF_DE.cu:913)
        const float o2 = __shfl_xor(s2, 32);
        const float C = s2 + o2;
        const float q = S / Df;
        const float r = sqrtf(q);
        const float a = (float)(-0.2 * (double)r);
        const float t1 = -20.0f * exp_f(a);
        const float c2 = C / Df;
        const float e2 = exp_f(c2);
        float u = t1 - e2;
        u = u + 20.0f;
        return (float)((double)u + 2.718282);
    } else if constexpr (FUNC == F_REF_GRIEWANK) {
        // 1 + S / 4000 - prod (the halves' partial products multiplied once)
        const float o2 = __shfl_xor(s2, 32);
        const float P = s2 * o2;
        const float s4 = S / 4000.0f;
        const float u = 1.0f + s4;
        return u - P;
    } else if constexpr (FUNC == F_REF_WEIERSTRASS) {
        // sum - D W with the reference's constant W in the task table
        const float dw = Df * tab[0];
        return S - dw;
    } else {
        return S;
    }
}

template <int NT, int FUNC, bool SKIP = false, bool ZPAD = false>
__device__ __forceinline__ float objective(const f16v (&acc)[NT], int D, const float* tab, int h) {
    // the row mask's bound: with ZPAD one no row reaches
    const int Dm = (ZPAD && zero_term_at_zero<FUNC>()) ? 0x7FFFFFFF : D;
    float s1 = 0.0f, s2 = (FUNC == F_REF_GRIEWANK) ? 1.0f : 0.0f;
    if constexpr (FUNC == F_ROSENBROCK) {
        float nb[NT][4];
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
            for (int g = 0; g < 4; ++g) nb[jt][g] = __shfl_xor(acc[jt][4 * g], 32);
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int j = 32 * jt + 8 * (r >> 2) + 4 * h + (r & 3);
                const int g = r >> 2;
                float zn;
                if ((r & 3) != 3) zn = acc[jt][r + 1];
                else if (g < 3) zn = h ? nb[jt][g + 1] : nb[jt][g];
                else zn = h ? ((jt + 1 < NT) ? nb[(jt + 1) % NT][0] : 0.0f) : nb[jt][g];
                const float z = acc[jt][r];
                const float zz = z * z;
                const float a = zz - zn;
                const float b = z - 1.0f;
                float t1 = 100.0f * a;
                t1 = t1 * a;
                const float b2 = b * b;
                const float v = t1 + b2;
                if (j + 1 < D) s1 = s1 + v;
            }
    } else if constexpr (FUNC == F_WEIERSTRASS && SKIP && !ZPAD) {
        // The wide kernels (SKIP, rows not zero-padded): four rows at a time, their terms
        // by the branch-free path (independent chains the scheduler interleaves), the rare
        // arguments redone by the full term, then the row sums in row order as below (s1 is
        // never -0, so adding +0 for a masked row leaves it).  The LDS epoch kernel keeps
        // one row at a time: there the interleaved chains take issue slots from the tasks
        // that share the CU and the mixed epoch is slower.
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (32 * jt + 8 * g >= D) continue;
                float v[4];
                bool rare = false;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float a = __builtin_fabsf(acc[jt][4 * g + e]);
                    const bool lo = a >= 2.32830644e-10f, hi = a >= 8388608.0f;
                    v[e] = weier_core(a, lo && !hi);
                    rare = rare || (!lo && !hi && a != 0.0f);  // NaN or 0 < |z| < 2^-32
                }
                if (rare) {
                    // one inlined copy of the full term: a rolled loop, the row picked by selects
#pragma unroll 1
                    for (int e = 0; e < 4; ++e) {
                        float z = acc[jt][4 * g];
                        z = e == 1 ? acc[jt][4 * g + 1] : z;
                        z = e == 2 ? acc[jt][4 * g + 2] : z;
                        z = e == 3 ? acc[jt][4 * g + 3] : z;
                        const float a = __builtin_fabsf(z);
                        if (z != z || (a > 0.0f && a < 2.32830644e-10f)) {
                            const float r = weier_rare(z);
#pragma unroll
                            for (int f = 0; f < 4; ++f) v[f] = e == f ? r : v[f];
                        }
                    }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int j = 32 * jt + 8 * g + 4 * h + e;
                    s1 = s1 + (j < Dm ? v[e] : 0.0f);
                }
            }
    } else {
        // SKIP: groups of eight rows past the dimension are skipped outright (a
        // uniform branch) for the objectives with transcendental terms -- worth it
        // where the row tiles are padded far past D (the wide kernel) or the terms are
        // costly (Weierstrass, Schwefel in the LDS kernel); rows j >= D are masked in
        // every case
        constexpr bool skip = SKIP && FUNC != F_SPHERE && FUNC != F_ELLIPTIC;
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (skip && 32 * jt + 8 * (r >> 2) >= D) continue;
                const int j = 32 * jt + 8 * (r >> 2) + 4 * h + (r & 3);
                const float z = acc[jt][r];
                if constexpr (FUNC == F_SPHERE) {
                    const float v = z * z;
                    if (j < Dm) s1 = s1 + v;
                } else if constexpr (FUNC == F_ELLIPTIC) {
                    const float zz = z * z;
                    const float v = tab[j] * zz;
                    if (j < Dm) s1 = s1 + v;
                } else if constexpr (FUNC == F_ACKLEY) {
                    const float v = z * z;
                    const float sq = sinpi_sq(z);
                    if (j < Dm) { s1 = s1 + v; s2 = s2 + sq; }
                } else if constexpr (FUNC == F_RASTRIGIN) {
                    const float zz = z * z;
                    const float s20 = 20.0f * sinpi_sq(z);
                    const float v = zz + s20;
                    if (j < Dm) s1 = s1 + v;
                } else if constexpr (FUNC == F_GRIEWANK) {
                    const float v = z * z;
                    const float a = 2.0f * sinpi_sq(z * tab[j]);
                    if (j < Dm) {
                        s1 = s1 + v;
                        const float om = 1.0f - s2;
                        const float aq = a * om;
                        s2 = s2 + aq;
                    }
                } else if constexpr (FUNC == F_WEIERSTRASS) {
                    if (j < Dm) s1 = s1 + weier_term(z);
                } else if constexpr (FUNC == F_SCHWEFEL) {
                    const float sq = sqrtf(__builtin_fabsf(z));
                    const float tv = sq * 0.159154937f;
                    const float v = z * sin2pi(tv);
                    if (j < Dm) s1 = s1 + v;
                } else if constexpr (FUNC == F_REF_ACKLEY) {
                    // the reference's terms: z^2 and cospif(2 z)
                    const float v = z * z;
                    const float tz = 2.0f * z;
                    const float c = cospi_f(tz);
                    if (j < Dm) { s1 = s1 + v; s2 = s2 + c; }
                } else if constexpr (FUNC == F_REF_RASTRIGIN) {
                    // z^2 - 10 cospif(2 z) + 10
                    const float zz = z * z;
                    const float tz = 2.0f * z;
                    const float c = cospi_f(tz);
                    const float t = 10.0f * c;
                    float v = zz - t;
                    v = v + 10.0f;
                    if (j < Dm) s1 = s1 + v;
                } else if constexpr (FUNC == F_REF_GRIEWANK) {
                    // z^2 and the factor cosf(z / sqrtf(j + 1)), cos q = 1 - 2 sin^2(q / 2)
                    const float v = z * z;
                    const float q = z / tab[j];
                    const float tq = q * 0.159154937f;
                    const float t = 2.0f * sinpi_sq(tq);
                    const float c = 1.0f - t;
                    if (j < Dm) { s1 = s1 + v; s2 = s2 * c; }
                } else if constexpr (FUNC == F_REF_WEIERSTRASS) {
                    if (j < Dm) s1 = s1 + weier_ref_term(z);
                }
            }
    }
    return objective_tail<FUNC>(s1, s2, D, tab, h);
}

// One 32-row tile (tile jt, accumulators acc) of the objective, in two parts: the row
// terms (independent of every other tile; zn0: Rosenbrock's z of row 32 (jt + 1) for this
// column, 0 past the last tile), then their sums onto the lane's running s1, s2 -- the
// rows of tile jt in the order objective() adds them.
template <int FUNC>
__device__ __forceinline__ void tile_vals(const f16v& acc, int jt, int D, const float* tab, int h, float zn0,
                                          float (&v1)[16], float (&v2)[16]) {
    if constexpr (FUNC == F_ROSENBROCK) {
        float nb[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) nb[g] = __shfl_xor(acc[4 * g], 32);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int g = r >> 2;
            float zn;
            if ((r & 3) != 3) zn = acc[r + 1];
            else if (g < 3) zn = h ? nb[g + 1] : nb[g];
            else zn = h ? zn0 : nb[g];
            v1[r] = rosen_val(acc[r], zn);
            v2[r] = 0.0f;
        }
    } else if constexpr (FUNC == F_WEIERSTRASS) {
        // four rows at a time through the branch-free term (as in the wide kernels'
        // objective), groups of eight rows past D skipped (a uniform branch); v1 = 0 for the
        // masked rows as row_vals gives
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v1[4 * g + e] = 0.0f;
                v2[4 * g + e] = 0.0f;
            }
            if (32 * jt + 8 * g >= D) continue;
            float v[4];
            bool rare = false;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a = __builtin_fabsf(acc[4 * g + e]);
                const bool lo = a >= 2.32830644e-10f, hi = a >= 8388608.0f;
                v[e] = weier_core(a, lo && !hi);
                rare = rare || (!lo && !hi && a != 0.0f);  // NaN or 0 < |z| < 2^-32
            }
            if (rare) {
#pragma unroll 1
                for (int e = 0; e < 4; ++e) {
                    float z = acc[4 * g];
                    z = e == 1 ? acc[4 * g + 1] : z;
                    z = e == 2 ? acc[4 * g + 2] : z;
                    z = e == 3 ? acc[4 * g + 3] : z;
                    const float a = __builtin_fabsf(z);
                    if (z != z || (a > 0.0f && a < 2.32830644e-10f)) {
                        const float r = weier_rare(z);
#pragma unroll
                        for (int f = 0; f < 4; ++f) v[f] = e == f ? r : v[f];
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = 32 * jt + 8 * g + 4 * h + e;
                v1[4 * g + e] = j < D ? v[e] : 0.0f;
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            v1[r] = 0.0f;
            v2[r] = 0.0f;
            row_vals<FUNC>(acc[r], 32 * jt + 8 * (r >> 2) + 4 * h + (r & 3), D, tab, v1[r], v2[r]);
        }
    }
}

template <int FUNC>
__device__ __forceinline__ void tile_sums(const float (&v1)[16], const float (&v2)[16], int jt, int D, int h, float& s1,
                                          float& s2) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int j = 32 * jt + 8 * (r >> 2) + 4 * h + (r & 3);
        if constexpr (FUNC == F_ROSENBROCK) {
            if (j + 1 < D) s1 = s1 + v1[r];
        } else {
            row_sum<FUNC>(v1[r], v2[r], j < D, s1, s2);
        }
    }
}

// Per-point factors of d f / d z: Ackley's two (from the sums over the point's z).
struct DzConst {
    float ka, kb;
};

// Ackley's gradient factors from its sums s1 = sum z_j^2, s2 = sum sin^2(pi z_j).
__device__ __forceinline__ DzConst ackley_const(float s1, float s2, int D) {
    DzConst k;
    const float Df = (float)D;
    const float r = sqrtf(s1 / Df);
    const float e1 = expm1_f(-0.2f * r) + 1.0f;
    const float e2 = expm1_f(-2.0f * (s2 / Df)) + 1.0f;
    k.ka = (r > 0.0f) ? (4.0f * e1) / (Df * r) : 0.0f;
    k.kb = (6.28318548f * 2.71828175f / Df) * e2;
    return k;
}

// Griewank's factor cos(theta_j) = 1 - 2 sin^2(theta_j / 2), theta_j / (2 pi) = z_j tab[j]
__device__ __forceinline__ float griewank_cos(float zj, float tj) { return 1.0f - 2.0f * sinpi_sq(zj * tj); }

// d f / d z_j for j < D of a point: zj = z_j, zp / zn = z_{j-1} / z_{j+1} (Rosenbrock only,
// ignored where the row does not exist), tj the row's table entry; Griewank takes
// pre = prod_{k<j} cos(theta_k) and suf = prod_{k>j} cos(theta_k), accumulated from the top.
template <int FUNC>
__device__ __forceinline__ float dz_elem(int j, float zj, float zp, float zn, int D, float tj, const DzConst& kc,
                                         float pre, float suf) {
    float v = 0.0f;
    if constexpr (FUNC == F_SPHERE) v = 2.0f * zj;
    else if constexpr (FUNC == F_ELLIPTIC) v = 2.0f * tj * zj;
    else if constexpr (FUNC == F_RASTRIGIN) v = 2.0f * zj + 62.8318531f * sin2pi(zj);
    else if constexpr (FUNC == F_ACKLEY) v = kc.ka * zj + kc.kb * sin2pi(zj);
    else if constexpr (FUNC == F_ROSENBROCK) {
        if (j + 1 < D) v = 400.0f * zj * (zj * zj - zn) + 2.0f * (zj - 1.0f);
        if (j > 0) v = v - 200.0f * (zp * zp - zj);
    } else if constexpr (FUNC == F_GRIEWANK) {
        const float sn = sin2pi(zj * tj);  // sin(theta_j)
        v = zj / 2000.0f + pre * suf * sn * (6.28318548f * tj);
    } else if constexpr (FUNC == F_WEIERSTRASS) {
        // sum_k 2^(1-k) pi 3^k sin(2 pi 3^k z), fractions of 3^k |z| as in the forward pass
        const float a = __builtin_fabsf(zj);
        float acc = 0.0f;
        if (a < 8388608.0f) {
            float c = 6.28318548f;  // 2 pi (1.5)^k
            if (a < 2.32830644e-10f) {
                float p3 = 1.0f;
                for (int k = 0; k <= 20; ++k) {
                    acc = fmaf(c, sin2pi(a * p3), acc);
                    c = c * 1.5f;
                    p3 = p3 * 3.0f;
                }
            } else {
                const uint32_t u = __float_as_uint(a);
                const int ex = (int)((u >> 23) & 0xFFu) - 127;
                const uint64_t m = (uint64_t)((u & 0x007FFFFFu) | 0x00800000u);
                uint64_t y = m << (64 - (23 - ex));
                for (int k = 0; k <= 20; ++k) {
                    const float r = (float)(uint32_t)(y >> 32) * 2.3283064365386963e-10f;
                    acc = fmaf(c, sin2pi(r), acc);
                    c = c * 1.5f;
                    y = y + (y << 1);
                }
            }
        }
        v = __builtin_copysignf(1.0f, zj) * acc;
    } else if constexpr (FUNC == F_SCHWEFEL) {
        const float sq = sqrtf(__builtin_fabsf(zj));
        const float t = sq * 0.159154937f;
        v = -(sin2pi(t) + 0.5f * sq * sin2pi(t + 0.25f));
    }
    return v;
}

}  // namespace emtf
