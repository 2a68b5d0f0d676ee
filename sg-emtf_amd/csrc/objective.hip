// objective.hip -- the stand-alone objective and its adjoint (emtf_objective_fwd /
// emtf_objective_adjoint) on gfx950: f = f(Q (x - o)) and gx = gf Q^T (df/dz) for n points.
//
// A wave evaluates 32 points: z = Q (x - o) by v_mfma_f32_32x32x2_f32 (A = Q from LDS, B = 32
// points, one per column, one gene parity per lane half), each lane left with 16 rows of z
// of its own point per 32-row tile -- the engine's evaluator, the same fma chains and sums,
// so the same bits.  The adjoint stays in registers from there: df/dz replaces z row by row,
// one half-wave swap per pair of rows turns the accumulator layout into the B operand of the
// second contraction gx = Q^T dz (A = Q read by columns), and gx leaves through the wave's
// LDS strip so that rows are stored whole.
//
// What bounds it: the FP32 MFMA (2 n D^2 operations forward, 4 n D^2 adjoint, rows padded
// to 32) with the points' memory traffic behind it.  So Q is staged once per workgroup, which
// then takes tile after tile, the points come through a per-wave strip of 32 genes
// (coalesced, the next strip's loads in flight during the current one's MFMA steps), and
// nothing is kept per point in LDS, so that at least two waves share a SIMD.  Against a build
// that staged Q again for every 128 points and kept the rows in LDS: 2^20 points of D = 50
// (Ackley) 229 to 99 us (53 TFLOP/s), 99991 of D = 200 (Schwefel) 404 to 130 us (62), value and
// gradient of 250000 of D = 100 (Griewank) 3170 to 295 us (51).
//
// NT = 1 .. 4 (dim <= 128): Q resident in LDS.  NT = 5 .. 8, forward only: Q does not fit,
// its 32-gene column strip is staged beside the points' and double buffered.
#include <hip/hip_runtime.h>
#include "emtf_eval.h"
#include "emtf_math.h"
#include "emtf_types.h"

#if !defined(EMTF_OBJ_NT)
#error "compile with -DEMTF_OBJ_NT=<32-row tiles, 1..8>"
#endif

namespace emtf {

constexpr int kCW = 32;       // genes per strip
constexpr int kCS = kCW + 4;  // LDS stride of a strip row: [16 even | 16 odd genes] + 4
constexpr int kCus = 256;     // compute units

// Threads per workgroup: the Q image is shared by more waves where it is large, so that two
// waves share a SIMD at every dimension (NT = 4: 67 KB of Q, 8 x 4.6 KB of strips).
template <int NT>
constexpr int obj_threads() { return NT >= 3 ? 512 : 256; }

// One strip of the wave's 32 points in flight.  Lane -> gene (lane & (w - 1)) of the strip,
// rows (lane / w) + i (64 / w), w = 2^LW genes: 32, or the whole row where it is short.
// x: the tile's first point (uniform); last: the last point the tile may read, which the rows
// past the batch repeat (their results are not stored).
template <int LW>
__device__ __forceinline__ void strip_load(float (&v)[1 << (LW - 1)], const ObjArgs& a, int tile, int c, int lane) {
    const int D = a.dim;
    const float* x = a.x + (int64_t)tile * 32 * D;
    const int rest = a.n - 1 - tile * 32;
    // the lane index is made opaque: masks and offsets derived from it are not kept in
    // registers from strip to strip
    asm volatile("" : "+v"(lane));
    const int d = kCW * c + (lane & ((1 << LW) - 1));
    const unsigned top = (unsigned)(rest < 31 ? rest : 31) * (unsigned)D + (unsigned)d;
    unsigned off = (unsigned)(lane >> LW) * (unsigned)D + (unsigned)d;
    const unsigned step = (unsigned)(64 >> LW) * (unsigned)D;
    if (d < D) {
#pragma unroll
        for (int i = 0; i < (1 << (LW - 1)); ++i) {
            v[i] = x[off < top ? off : top];
            off += step;
        }
    }
}

// w = x - o into the wave's strip buffer (zero past the dimension).
template <int LW>
__device__ __forceinline__ void strip_store(float* buf, const float (&v)[1 << (LW - 1)], const float* o_s, int D, int c,
                                            int lane) {
    asm volatile("" : "+v"(lane));
    const int gl = lane & ((1 << LW) - 1), d = kCW * c + gl;
    const bool in = d < D;
    const float o = o_s[d];
    float* p = buf + (lane >> LW) * kCS + (gl & 1) * (kCW / 2) + (gl >> 1);
#pragma unroll
    for (int i = 0; i < (1 << (LW - 1)); ++i) p[i * (64 >> LW) * kCS] = in ? v[i] - o : 0.0f;
}

// 2^LW genes (from 32 c) of the tile's gradient rows (`rows` of them) out of the strip buffer.
template <int LW>
__device__ __forceinline__ void strip_out(float* gx, const float* buf, int rows, int D, int c, int lane) {
    asm volatile("" : "+v"(lane));
    const int gl = lane & ((1 << LW) - 1), row0 = lane >> LW, d = kCW * c + gl;
    unsigned off = (unsigned)row0 * (unsigned)D + (unsigned)d;
    const unsigned step = (unsigned)(64 >> LW) * (unsigned)D;
    const float* p = buf + row0 * kCS + gl;
#pragma unroll
    for (int i = 0; i < (1 << (LW - 1)); ++i) {
        if (d < D && row0 + i * (64 >> LW) < rows) gx[off] = p[i * (64 >> LW) * kCS];
        off += step;
    }
}

// a = (own lower half, other's lower half), b = (own upper's ..): a's upper 32 lanes and b's
// lower 32 lanes exchanged.
__device__ __forceinline__ void swap_halves(float& a, float& b) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r.x);
    b = __uint_as_float(r.y);
}

#if EMTF_OBJ_NT <= 4
// df/dz in the accumulator layout: z (rows j = 32 jt + 8 g + 4 h + e of the lane's point in
// z[jt][4 g + e]) becomes dz.
template <int NT, int FUNC>
__device__ __forceinline__ void dz_rows(f16v (&z)[NT], int D, const float* tab, int h) {
    DzConst kc{0.0f, 0.0f};
    if constexpr (FUNC == F_ACKLEY) {
        // sums over the dimensions in their order: the lower half-wave adds the z^2, the
        // upper one the sin^2, of both halves' rows
        float s = 0.0f;
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (32 * jt + 8 * g >= D) continue;
                float u[4], w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bool in = 32 * jt + 8 * g + 4 * h + e < D;
                    const float zj = z[jt][4 * g + e];
                    u[e] = in ? zj * zj : 0.0f;
                    w[e] = in ? sinpi_sq(zj) : 0.0f;
                    swap_halves(u[e], w[e]);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) s = s + u[e];
#pragma unroll
                for (int e = 0; e < 4; ++e) s = s + w[e];
            }
        float s1 = s, s2 = s;
        swap_halves(s1, s2);
        kc = ackley_const(s1, s2, D);
    }
    float pre[FUNC == F_GRIEWANK ? NT : 1][16];
    float suf = 1.0f;
    if constexpr (FUNC == F_GRIEWANK) {
        // prefix products over the dimensions in their order, each lane through both
        // halves' factors (1 past the dimension), kept for its own rows
        float p = 1.0f;
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (32 * jt + 8 * g >= D) continue;
                float lo[4], hi[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int j = 32 * jt + 8 * g + 4 * h + e;
                    lo[e] = j < D ? griewank_cos(z[jt][4 * g + e], tab[j]) : 1.0f;
                    hi[e] = lo[e];
                    swap_halves(lo[e], hi[e]);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    pre[jt][4 * g + e] = p;
                    p = p * lo[e];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    pre[jt][4 * g + e] = h ? p : pre[jt][4 * g + e];
                    p = p * hi[e];
                }
            }
    }
    float zup = 0.0f;  // Rosenbrock: z_{j+1} of the lane's last row of a group, from above
    // from the top: the suffix products run downwards, Rosenbrock's neighbours are read
    // before they are overwritten
    (void)zup;
#pragma unroll
    for (int jt = NT - 1; jt >= 0; --jt)
#pragma unroll
        for (int g = 3; g >= 0; --g) {
            const int j0 = 32 * jt + 8 * g;
            float sf[4] = {1.0f, 1.0f, 1.0f, 1.0f};
            float below = 0.0f, above = 0.0f;  // z_{j0 + 4 h - 1}, z_{j0 + 4 h + 4}
            if constexpr (FUNC == F_ROSENBROCK) {
                // first rows of this group (lower half's z_{j0}, upper half's z_{j0+4}) and the
                // upper half's last row of the group below, exchanged between the halves
                const float other0 = __shfl_xor(z[jt][4 * g], 32);
                const float other3 = __shfl_xor(z[jt][4 * g + 3], 32);
                above = h ? zup : other0;
                const float b3 = g > 0 ? z[jt][4 * g - 1] : (jt > 0 ? z[jt > 0 ? jt - 1 : 0][15] : 0.0f);
                const float ob3 = __shfl_xor(b3, 32);
                below = h ? other3 : ob3;
                zup = other0;  // the upper half's next group down ends below this z_{j0}
            }
            if constexpr (FUNC == F_GRIEWANK) {
                if (j0 < D) {
                    float lo[4], hi[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int j = j0 + 4 * h + e;
                        lo[e] = j < D ? griewank_cos(z[jt][4 * g + e], tab[j]) : 1.0f;
                        hi[e] = lo[e];
                        swap_halves(lo[e], hi[e]);
                    }
#pragma unroll
                    for (int e = 3; e >= 0; --e) {
                        sf[e] = suf;
                        suf = suf * hi[e];
                    }
#pragma unroll
                    for (int e = 3; e >= 0; --e) {
                        sf[e] = h ? sf[e] : suf;
                        suf = suf * lo[e];
                    }
                }
            }
            float out[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = j0 + 4 * h + e;
                const float zj = z[jt][4 * g + e];
                const float zp = e > 0 ? z[jt][4 * g + (e > 0 ? e - 1 : 0)] : below;
                const float zn = e < 3 ? z[jt][4 * g + (e < 3 ? e + 1 : 3)] : above;
                float v = 0.0f;
                if (j0 < D) {
                    const float tj = (FUNC == F_ELLIPTIC || FUNC == F_GRIEWANK) ? tab[j] : 0.0f;
                    v = dz_elem<FUNC>(j, zj, zp, zn, D, tj, kc, FUNC == F_GRIEWANK ? pre[FUNC == F_GRIEWANK ? jt : 0][4 * g + e] : 0.0f,
                                      sf[e]);
                }
                out[e] = j < D ? v : 0.0f;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) z[jt][4 * g + e] = out[e];
        }
}

// Q resident: LDS holds the Q image (32 NT rows of stride RS = 2 HS + 4, genes [even | odd],
// zero past the dimension; HS = Dh rounded up to 4), the shift, the table and one strip per
// wave.  Workgroups take tiles of 32 points per wave, grid-stride.
template <int NT, int LW, int FUNC, bool ADJ>
__global__ __launch_bounds__(obj_threads<NT>()) void objective_kernel(ObjArgs a, int tiles) {
    constexpr int THR = obj_threads<NT>(), NW = THR / 64;
    extern __shared__ __align__(16) float smem[];
    const int D = a.dim, Dh = (D + 1) >> 1, HS = (Dh + 3) & ~3, RS = 2 * HS + 4;
    float* Q = smem;
    float* o_s = Q + 32 * NT * RS;
    float* tab = o_s + 32 * NT;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 31, h = lane >> 5;
    float* buf = tab + 32 * NT + wave * 32 * kCS;
    for (int e = tid; e < 32 * NT * RS; e += THR) Q[e] = 0.0f;
    for (int d = tid; d < 32 * NT; d += THR) {
        o_s[d] = (d < D && a.shift) ? a.shift[d] : 0.0f;
        tab[d] = d < D ? a.tab[d] : 0.0f;
    }
    __syncthreads();
    if (a.has_rot) {
        // eight loads in flight per thread
        const int total = D * D;
        for (int e0 = tid; e0 < total; e0 += 8 * THR) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int e = e0 + k * THR;
                v[k] = a.rot[e < total ? e : 0];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int e = e0 + k * THR;
                if (e < total) {
                    const int j = e / D, d = e - j * D;
                    Q[j * RS + (d & 1) * HS + (d >> 1)] = v[k];
                }
            }
        }
    } else {
        for (int d = tid; d < D; d += THR) Q[d * RS + (d & 1) * HS + (d >> 1)] = 1.0f;
    }
    __syncthreads();
    const int nc = (D + kCW - 1) / kCW;
    const int stride = gridDim.x * NW;
    int tile = blockIdx.x * NW + wave;
    float v[1 << (LW - 1)] = {};
    if (tile < tiles) strip_load<LW>(v, a, tile, 0, lane);
    const float* qrow = Q + col * RS + h * HS;
    const float* brow = buf + col * kCS + h * (kCW / 2);
    for (; tile < tiles; tile += stride) {
        const int pt0 = tile * 32;
        f16v acc[NT];
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[jt][r] = 0.0f;
#pragma unroll 1
        for (int c = 0; c < nc; ++c) {
            wave_lds_fence();  // the strip's previous readers are done
            strip_store<LW>(buf, v, o_s, D, c, lane);
            wave_lds_fence();
            if (c + 1 < nc) strip_load<LW>(v, a, tile, c + 1, lane);
            else if (tile + stride < tiles) strip_load<LW>(v, a, tile + stride, 0, lane);
            const int left = Dh - 16 * c, nb = left >= 16 ? 4 : (left + 3) >> 2;  // blocks of four k-steps
#pragma unroll 1
            for (int b = 0; b < nb; ++b) {
                const float4 w = lds4(brow + 4 * b);
                float4 q[NT];
#pragma unroll
                for (int jt = 0; jt < NT; ++jt) q[jt] = lds4(qrow + 32 * jt * RS + 16 * c + 4 * b);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int jt = 0; jt < NT; ++jt)
                        acc[jt] = __builtin_amdgcn_mfma_f32_32x32x2f32(f4(q[jt], e), f4(w, e), acc[jt], 0, 0, 0);
            }
        }
        const int pt = pt0 + col;
        const bool valid = pt < a.n;
        // row masks and table addresses derived from the half index stay out of the loop's registers
        int hh = h;
        asm volatile("" : "+v"(hh));
        if constexpr (!ADJ) {
            const float f = objective<NT, FUNC, true>(acc, D, tab, hh);
            if (valid && h == 0) a.f[pt] = f;
        } else {
            const float up = a.gf[valid ? pt : a.n - 1];
            dz_rows<NT, FUNC>(acc, D, tab, hh);
            f16v gacc[NT];
#pragma unroll
            for (int dt = 0; dt < NT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) gacc[dt][r] = 0.0f;
            const float* qc = Q + h * RS + (col & 1) * HS + (col >> 1);  // row j0 + 2 e + h as the k-steps go
#pragma unroll
            for (int jt = 0; jt < NT; ++jt)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    if (32 * jt + 8 * g >= D) continue;
                    float k0 = acc[jt][4 * g] * up, k1 = acc[jt][4 * g + 2] * up;
                    float k2 = acc[jt][4 * g + 1] * up, k3 = acc[jt][4 * g + 3] * up;
                    swap_halves(k0, k2);  // rows j0, j0 + 1 | j0 + 4, j0 + 5
                    swap_halves(k1, k3);  // rows j0 + 2, j0 + 3 | j0 + 6, j0 + 7
                    const float kk[4] = {k0, k1, k2, k3};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
#pragma unroll
                        for (int dt = 0; dt < NT; ++dt)
                            gacc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(qc[16 * dt], kk[e], gacc[dt], 0, 0, 0);
                        qc += 2 * RS;
                        // one address stepped, not one kept in a register per k-step
                        asm volatile("" : "+v"(qc));
                    }
                }
            // 32 genes of the 32 points at a time through the wave's strip
#pragma unroll
            for (int dt = 0; dt < NT; ++dt) {
                if (32 * dt >= D) continue;
                wave_lds_fence();
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<float4*>(buf + col * kCS + 8 * g + 4 * h) =
                        make_float4(gacc[dt][4 * g], gacc[dt][4 * g + 1], gacc[dt][4 * g + 2], gacc[dt][4 * g + 3]);
                wave_lds_fence();
                strip_out<LW>(a.gx + (int64_t)pt0 * D, buf, a.n - pt0, D, dt, lane);
            }
        }
    }
}
#else
// Q too large for LDS (forward only): per strip of 32 genes the workgroup stages Q's columns
// (32 NT rows, double buffered, the next strip's loads in flight during the MFMA steps), one
// barrier per strip; each wave its own points' strip.
constexpr int kWideThreads = 512;

template <int NT, int FUNC>
__global__ __launch_bounds__(kWideThreads) void objective_wide_kernel(ObjArgs a, int tiles) {
    constexpr int THR = kWideThreads, NW = THR / 64, QN = 32 * NT * kCS, NQ = 32 * NT * kCW / THR;
    extern __shared__ __align__(16) float smem[];
    const int D = a.dim, Dh = (D + 1) >> 1;
    float* Q = smem;  // two strips
    float* o_s = Q + 2 * QN;
    float* tab = o_s + 32 * NT;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 31, h = lane >> 5;
    float* buf = tab + 32 * NT + wave * 32 * kCS;
    for (int d = tid; d < 32 * NT; d += THR) {
        o_s[d] = (d < D && a.shift) ? a.shift[d] : 0.0f;
        tab[d] = d < D ? a.tab[d] : 0.0f;
    }
    __syncthreads();
    const int nc = (D + kCW - 1) / kCW, per = gridDim.x * NW;
    const int qg = tid & 31, qr = tid >> 5;  // the thread's gene of the strip, first row (rows qr + 16 i)
    float qv[NQ];
    auto q_load = [&](int c) {
        const int d = kCW * c + qg;
        unsigned off = (unsigned)(qr * D + d);
        asm volatile("" : "+v"(off));  // one offset stepped, not one kept in a register per row
        const unsigned step = (unsigned)(THR / 32 * D);
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const bool in = d < D && off < (unsigned)(D * D);  // row < D
            if (a.has_rot) qv[i] = in ? a.rot[off] : 0.0f;
            else qv[i] = in && qr + i * (THR / 32) == d ? 1.0f : 0.0f;
            off += step;
        }
    };
    auto q_store = [&](float* dst) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) dst[(qr + i * (THR / 32)) * kCS + (qg & 1) * (kCW / 2) + (qg >> 1)] = qv[i];
    };
    const float* brow = buf + col * kCS + h * (kCW / 2);
    // every wave goes through the same strips (the barriers); a wave past the last tile
    // repeats it and stores nothing
    float v[16] = {};
    int cur = 0;
    const int first = blockIdx.x * NW + wave;
    q_load(0);
    strip_load<5>(v, a, first < tiles ? first : tiles - 1, 0, lane);
    for (int base = blockIdx.x * NW; base < tiles; base += per) {
        const int tile = base + wave < tiles ? base + wave : tiles - 1;
        const int pt0 = tile * 32;
        f16v acc[NT];
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[jt][r] = 0.0f;
#pragma unroll 1
        for (int c = 0; c < nc; ++c) {
            q_store(Q + cur * QN);
            wave_lds_fence();
            strip_store<5>(buf, v, o_s, D, c, lane);
            __syncthreads();  // this strip's Q is staged; the other buffer's readers passed the last one
            const float* qrow = Q + cur * QN + col * kCS + h * (kCW / 2);
            if (c + 1 < nc) {
                q_load(c + 1);
                strip_load<5>(v, a, tile, c + 1, lane);
            } else if (base + per < tiles) {
                const int nt = base + per + wave < tiles ? base + per + wave : tiles - 1;
                q_load(0);
                strip_load<5>(v, a, nt, 0, lane);
            }
            const int left = Dh - 16 * c, nb = left >= 16 ? 4 : (left + 3) >> 2;
#pragma unroll 1
            for (int b = 0; b < nb; ++b) {
                const float4 w = lds4(brow + 4 * b);
                float4 q[NT];
#pragma unroll
                for (int jt = 0; jt < NT; ++jt) q[jt] = lds4(qrow + 32 * jt * kCS + 4 * b);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int jt = 0; jt < NT; ++jt)
                        acc[jt] = __builtin_amdgcn_mfma_f32_32x32x2f32(f4(q[jt], e), f4(w, e), acc[jt], 0, 0, 0);
            }
            cur ^= 1;
        }
        int hh = h;
        asm volatile("" : "+v"(hh));
        const float f = objective<NT, FUNC, true>(acc, D, tab, hh);
        const int pt = pt0 + col;
        if (base + wave < tiles && pt < a.n && h == 0) a.f[pt] = f;
    }
}
#endif

}  // namespace emtf

#define EMTF_OCAT2(a, b) a##b
#define EMTF_OCAT(a, b) EMTF_OCAT2(a, b)

// Workgroups of `nw` waves for `tiles` tiles: as many as are resident at `lds` bytes each
// (two waves a SIMD of these register counts), fewer where every one of them takes the same
// number of tiles.
static int obj_grid(int tiles, int nw, int lds) {
    const int wgs = (tiles + nw - 1) / nw;
    int occ = 160 * 1024 / lds;
    const int most = 16 / nw;
    occ = occ < 1 ? 1 : (occ < most ? occ : most);
    const int slots = emtf::kCus * occ;
    const int rounds = (wgs + slots - 1) / slots;
    return (wgs + rounds - 1) / rounds;
}

template <typename K>
static hipError_t obj_launch(K k, const emtf::ObjArgs& a, int threads, int lds, hipStream_t stream) {
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
    }
    const int tiles = (int)(((int64_t)a.n + 31) / 32);
    hipLaunchKernelGGL(k, dim3(obj_grid(tiles, threads / 64, lds)), dim3(threads), lds, stream, a, tiles);
    return hipGetLastError();
}

template <int FUNC>
static hipError_t obj_any(const emtf::ObjArgs& a, int adjoint, hipStream_t s) {
    constexpr int NT = EMTF_OBJ_NT;
    using namespace emtf;
#if EMTF_OBJ_NT <= 4
    constexpr int THR = obj_threads<NT>();
    const int HS = (((a.dim + 1) >> 1) + 3) & ~3;
    const int lds = 4 * (32 * NT * (2 * HS + 4) + 64 * NT + (THR / 64) * 32 * kCS);
    // rows of at most 8 or 16 genes: a load instruction takes 8 or 4 of them
#if EMTF_OBJ_NT == 1
    if (a.dim <= 8)
        return adjoint ? obj_launch(&objective_kernel<NT, 3, FUNC, true>, a, THR, lds, s)
                       : obj_launch(&objective_kernel<NT, 3, FUNC, false>, a, THR, lds, s);
    if (a.dim <= 16)
        return adjoint ? obj_launch(&objective_kernel<NT, 4, FUNC, true>, a, THR, lds, s)
                       : obj_launch(&objective_kernel<NT, 4, FUNC, false>, a, THR, lds, s);
#endif
    return adjoint ? obj_launch(&objective_kernel<NT, 5, FUNC, true>, a, THR, lds, s)
                   : obj_launch(&objective_kernel<NT, 5, FUNC, false>, a, THR, lds, s);
#else
    if (adjoint) return hipErrorInvalidValue;
    const int lds = 4 * (2 * 32 * NT * kCS + 64 * NT + (kWideThreads / 64) * 32 * kCS);
    return obj_launch(&objective_wide_kernel<NT, FUNC>, a, kWideThreads, lds, s);
#endif
}

// emtf_launch_objective_nt<NT>: dims up to 32 NT (adjoint: NT <= 4).
extern "C" int EMTF_OCAT(emtf_launch_objective_nt, EMTF_OBJ_NT)(const emtf::ObjArgs* a, int adjoint, hipStream_t s) {
    switch (a->func) {
    case 0: return (int)obj_any<0>(*a, adjoint, s);
    case 1: return (int)obj_any<1>(*a, adjoint, s);
    case 2: return (int)obj_any<2>(*a, adjoint, s);
    case 3: return (int)obj_any<3>(*a, adjoint, s);
    case 4: return (int)obj_any<4>(*a, adjoint, s);
    case 5: return (int)obj_any<5>(*a, adjoint, s);
    case 6: return (int)obj_any<6>(*a, adjoint, s);
    case 7: return (int)obj_any<7>(*a, adjoint, s);
    }
    return (int)hipErrorInvalidValue;
}
