// cvrp.hip -- capacitated-VRP genetic algorithm on gfx950 (exact integer arithmetic).
//
// One workgroup of eight waves owns one instance for an epoch of generations.  Everything an
// epoch touches lives in LDS: two giant tours (uint8 customer ids) per individual, of which
// one is the individual and the other its child, and the nodes (coordinates relative to
// the depot, depot distance, demand).  Distances between customers are computed when needed:
// nint(sqrt(dx^2 + dy^2)) of integer differences is exact in binary32 (sqrt of an integer
// <= 65280 lies at least 4.9e-4 from every half-integer, far above the square root's
// rounding).  A generation goes through the individuals 64 at a time:
//   1. a wave per individual, a lane per position: mate, cut points and mutation from Philox
//      (lane q of a wave draws for the wave's q-th individual), the child by Davis order
//      crossover (OX) with the swap / 2-opt mutation folded into where a gene is written, then
//      what the split needs of it: per position the saving of joining it to its
//      predecessor's route and the length of its window (a demand scan and a binary search);
//   2. four lanes per individual: the Prins split (shortest path over the giant tour, routes
//      of load <= capacity) as a sliding-window minimum held in registers;
//   3. the child replaces its parent iff its cost is <= the parent's (reference Selection
//      rule, proposed model/SG-EMTF_cvrp.cu): the two tours change roles.
// What bounds it: the split is a serial chain of n steps per individual, so a step must be
// short, and everything that does not depend on the labels is taken out of it.  With one
// lane per individual doing all of it (64 times fewer waves, each waiting for its own LDS
// loads and for the wave's longest window move at every step) a generation of 200 customers
// took 150 us, now 63 (512 instances of 50 to 200 customers, pop 128, 100 generations: 15.1 to
// 6.3 ms; the split is a third of it).
// The reference's CVRP kernel (SG-EMTF_cvrp.cu:668-962) is a prototype whose
// crossover overwrites genomes with ones; this implements the algorithm it names.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "emtf_math.h"
#include "cvrp_types.h"

namespace emtf {

constexpr uint32_t P_CV_INIT = 16, P_CV_GEN = 17;
constexpr int kCvThreads = 512;  // eight waves: two workgroups of n = 200 share a CU; twice that
                                 // where a CU has one instance at most (emtf_cvrp_launch)
constexpr int kCvBatch = 64;     // individuals per pass
constexpr int kSlots = 16;       // window positions in registers; longer windows read the rest from LDS

// One row of split data per individual of a pass, in words: n + 1 entries, an odd number of
// words so that the rows of a wave start in different banks.
__host__ __device__ inline int cv_row_words(int n, int entry_bytes) {
    return (entry_bytes == 2 ? (n + 2) / 2 : n + 1) | 1;
}

// RowT: uint16_t entries (W + woff) when every instance's W + woff range fits 16 bits,
// else uint32_t.
template <typename RowT>
struct CvLds {
    RowT* G;        // kCvBatch rows of split data
    int32_t* cost;  // popP
    int32_t* ord;   // popP
    int32_t* aux;   // popP
    int32_t* cur;   // popP: bit 0 the tour that is the individual, bit 1 its child was accepted
    int32_t* info;  // kCvBatch: path length + last depot distance; negative: a window past kSlots
    uint2* node;    // n + 1: coordinates relative to the depot (x & 0xFFFF | y << 16), depot distance | demand << 8
    uint8_t* T;     // 2 x popP x NP tours
};

__host__ __device__ inline int cvrp_lds_bytes(int n, int popP, int entry_bytes) {
    const int NP = (n + 3) & ~3;
    return kCvBatch * cv_row_words(n, entry_bytes) * 4 + 4 * popP * 4 + kCvBatch * 4 + ((n + 1 + 1) & ~1) * 8 + 2 * popP * NP;
}

// TSPLIB EUC_2D distance nint(sqrt(dx^2 + dy^2)) of two packed relative coordinates.
// Every distance of an instance is <= 255 (checked at create), so s = dx^2 + dy^2 < 255.5^2,
// and sqrt(s) of an integer s lies at least 0.25 / 511 = 4.9e-4 from every half-integer;
// the hardware square root (v_sqrt_f32, 1 ulp <= 2^-16 below 256) and the rounding of
// the + 0.5 stay far inside that, so the rounded distance is exact without the
// correctly rounded square root's refinement.
// (Coordinate differences fit 16 bits: the nodes lie within 255.5 of the depot.)
typedef int16_t ss2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int nint_xy(uint32_t a, uint32_t b) {
    const ss2 d = __builtin_bit_cast(ss2, a) - __builtin_bit_cast(ss2, b);
    const int s = __builtin_amdgcn_sdot2(d, d, 0, false);
    return (int)(__builtin_amdgcn_sqrtf((float)s) + 0.5f);
}

// Inclusive sum over the wave's lanes: within rows of 16, then across them.
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, true);  // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, true);  // row_bcast:31 into rows 2 and 3
    return v;
}

// One individual's child in the making (uniform over its wave).
struct Breed {
    const uint8_t *p1, *p2;  // parents
    uint8_t* child;
    int a, b;                // p1's genes a .. b are taken
    int lo, span, hi, sum;   // mutation: position k with k - lo <= span (unsigned) or k == hi goes to sum - k
};

// The children of NI individuals (a wave makes them together: the LDS latencies of one
// are covered by the other's work), rows of n <= 64 NC genes, a lane per position: p1's genes
// at a .. b, then p2's other genes in order from b + 1 on, cyclically (OX), each written where
// the mutation leaves it.  rows[i]: scratch of n + 1 bytes (a flag per gene: taken from p1).
template <int NC, int NI>
__device__ __forceinline__ void make_children(const Breed (&bd)[NI], uint8_t* const (&rows)[NI], int n, int lane) {
    auto at = [&](const Breed& x, int k) {
        return (((unsigned)(k - x.lo) <= (unsigned)x.span) | (k == x.hi)) ? x.sum - k : k;
    };
    int g1[NI][NC], g2[NI][NC];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int s = 64 * c + lane < n ? 64 * c + lane : n - 1;  // lanes past the tour repeat its last gene
            const int q = bd[i].b + 1 + s;
            g1[i][c] = bd[i].p1[s];
            g2[i][c] = bd[i].p2[q < n ? q : q - n];
        }
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int s = 64 * c + lane < n ? 64 * c + lane : n - 1;
            const bool seg = (unsigned)(s - bd[i].a) <= (unsigned)(bd[i].b - bd[i].a);
            rows[i][g1[i][c]] = seg ? 1 : 0;
            if (seg) bd[i].child[at(bd[i], s)] = (uint8_t)g1[i][c];
        }
    wave_lds_fence();
    int taken[NI][NC];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) taken[i][c] = rows[i][g2[i][c]];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        int k0 = bd[i].b + 1;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const bool keep = (taken[i][c] == 0) & (64 * c + lane < n);
            const unsigned long long bal = __ballot(keep);
            const int k = __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, (unsigned)k0));
            if (keep) bd[i].child[at(bd[i], k < n ? k : k - n)] = (uint8_t)g2[i][c];
            k0 += __popcll(bal);
        }
    }
    wave_lds_fence();
}

// What the split of NI tours needs, a wave for all of them, a lane per position.  With path
// prefix sums P_k = sum_{m<k} d(t_m, t_{m+1}) the route t_i .. t_{j-1} costs
// d(0, t_i) + P_{j-1} - P_i + d(t_{j-1}, 0), so with W_i = V_i + d(0, t_i) - P_i the labels are
//   V_j = P_{j-1} + d(t_{j-1}, 0) + min W_i over the k_j starts i = j - k_j .. j - 1 whose
//   demand fits the capacity, and W_j = g_j + that minimum,
//   g_j = d(t_{j-1}, 0) + d(0, t_j) - d(t_{j-1}, t_j)
// -- the same integer sums and minimum as the pull form, so the same labels.  Entry p of the
// row: (g_p + 1) << 6 | k_{p+1} (g_0 = d(0, t_0); -1 <= g <= 510 by the triangle inequality of
// the rounded distances, 1 <= k <= 63).  info[i]: P_{n-1} + d(t_{n-1}, 0), its sign bit set when
// a window is longer than kSlots.  The windows by binary search in the demand prefix sums
// (kept in the row meanwhile): steps 16 .. 1 reach 32 starts, a second round for the rest.
template <int NC, int NI, typename RowT>
__device__ __forceinline__ void split_data(const uint8_t* const (&t)[NI], RowT* const (&row)[NI], int32_t* const (&info)[NI],
                                           const uint2* node, int n, int cap, int lane) {
    int cur[NI][NC], prv[NI][NC], S[NI][NC], g[NI][NC], q[NI][NC], path[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int p = 64 * c + lane < n ? 64 * c + lane : n - 1;
            cur[i][c] = t[i][p];
            prv[i][c] = c > 0 || lane > 0 ? t[i][c > 0 || lane > 0 ? p - 1 : 0] : 0;  // the depot before the first
        }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        path[i] = 0;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const bool in = 64 * c + lane < n;
            const uint2 v = node[cur[i][c]], u = node[prv[i][c]];
            int d = nint_xy(u.x, v.x);
            d = c == 0 && lane == 0 ? 0 : d;
            path[i] += in ? d : 0;
            g[i][c] = (int)((u.y & 0xFFu) + (v.y & 0xFFu)) - d;
            S[i][c] = wave_scan(in ? (int)(v.y >> 8) : 0);
            // the last lane of the tour holds the way back to the depot
            path[i] += 64 * c + lane == n - 1 ? (int)(v.y & 0xFFu) : 0;
        }
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        int carry = 0;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int last = __builtin_amdgcn_readlane(S[i][c], 63);
            S[i][c] += carry;  // demand of t_0 .. t_p
            carry += last;
            if (64 * c + lane < n) row[i][64 * c + lane + 1] = (RowT)S[i][c];
            q[i][c] = 64 * c + lane;  // the start found so far (one customer always fits)
        }
        if (lane == 0) row[i][0] = 0;
        path[i] = wave_scan(path[i]);
    }
    wave_lds_fence();
    auto search = [&]() {
#pragma unroll
        for (int w = 16; w >= 1; w >>= 1)
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    // a start i fits iff S_i >= S_j - cap; clamped to the first (if that fits, it is the start)
                    int x = q[i][c] - w;
                    x = x > 0 ? x : 0;
                    q[i][c] = (int)row[i][x] >= S[i][c] - cap ? x : q[i][c];
                }
    };
    search();
    bool more = false;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) more |= (64 * c + lane < n) & (64 * c + lane - q[i][c] == 31);
    if (__ballot(more)) search();
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        bool far = false;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int p = 64 * c + lane, k = p + 1 - q[i][c];
            far |= (p < n) & (k > kSlots);
            if (p < n) row[i][p] = (RowT)(((g[i][c] + 1) << 6) | k);
        }
        const bool any_far = __ballot(far) != 0;
        if (lane == 63) *info[i] = any_far ? (int)((uint32_t)path[i] | 0x80000000u) : path[i];
    }
}

typedef uint32_t __attribute__((may_alias)) u32a;
typedef uint16_t us2 __attribute__((ext_vector_type(2)));

// min over the four lanes of a quad
__device__ __forceinline__ int quad_min(int m) {
    const int a = __builtin_amdgcn_update_dpp(0, m, 0xB1, 0xF, 0xF, true);  // quad_perm:[1,0,3,2]
    m = a < m ? a : m;
    const int b = __builtin_amdgcn_update_dpp(0, m, 0x4E, 0xF, 0xF, true);  // quad_perm:[2,3,0,1]
    return b < m ? b : m;
}

// The split's recurrence over a row of split_data, four lanes per individual (sub: the lane's
// place in its quad): min W_i over the last window, + woff.  W_i sits in slot i mod 16: lane
// i & 3 of the quad, element (i >> 2) & 3 of the lane.  A step masks the slots that are older
// than the window (their ages at step u mod 16 are constants of the lane), takes the minimum
// in the lane, then over the quad, and the quad's lanes all hold the new W.  Four lanes: with
// one lane per individual a step is 32 instructions of a lone wave, with four it is 20
// and every SIMD of the CU has a wave of it.  FAR: windows past 16 exist; W is then also kept
// in the row (over the entry read before) and the older starts are read from there.
template <typename RowT, bool FAR>
struct SplitChain {
    static constexpr bool P16 = sizeof(RowT) == 2;
    static constexpr int NR = P16 ? 2 : 4;
    uint32_t w[NR], age[16][NR], k, nx, e2;
    bool own[4];
    RowT* row;
    int sub;

    __device__ __forceinline__ SplitChain(RowT* r, int s) : k(0), e2(0), row(r), sub(s) {
#pragma unroll
        for (int e = 0; e < 4; ++e) own[e] = sub == e;
#pragma unroll
        for (int r2 = 0; r2 < NR; ++r2) {
            w[r2] = 0xFFFFFFFFu;
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                // slot sub + 4 e was written 1 .. 16 steps before step u
                auto a = [&](int e) { return (uint32_t)((u - sub - 4 * e - 1) & 15) + 1u; };
                age[u][r2] = P16 ? (a(2 * r2) | (a(2 * r2 + 1) << 16)) : a(r2);
            }
        }
        nx = P16 ? reinterpret_cast<const u32a*>(row)[0] : row[0];  // a pair of entries (an entry) ahead
    }
    // the window's minimum before step j (u = j mod 16)
    __device__ __forceinline__ uint32_t minimum(int u, int j) {
        uint32_t m;
        if constexpr (P16) {
            const uint32_t kk = k | (k << 16);
            us2 c[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const ss2 d = __builtin_bit_cast(ss2, kk) - __builtin_bit_cast(ss2, age[u][r]);
                c[r] = __builtin_bit_cast(us2, (uint32_t)(w[r] | __builtin_bit_cast(uint32_t, (ss2)(d >> 15))));
            }
            const us2 q = __builtin_elementwise_min(c[0], c[1]);
            m = q.x < q.y ? q.x : q.y;
        } else {
            m = 0x7FFFFFFFu;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t c = age[u][r] <= k ? w[r] : 0x7FFFFFFFu;
                m = c < m ? c : m;
            }
        }
        if constexpr (FAR) {
            if (__ballot((int)k > kSlots)) {
                for (int i = j - kSlots - 1 - sub; i >= j - (int)k; i -= 4) {
                    const uint32_t v = row[i];
                    m = v < m ? v : m;
                }
            }
        }
        return (uint32_t)quad_min((int)m);
    }
    // W_j from the minimum; k becomes the next label's window
    __device__ __forceinline__ void advance(int u, int j, uint32_t m) {
        uint32_t gm, W;  // g, off the chain
        if constexpr (P16) {
            if ((u & 1) == 0) {
                e2 = nx;
                nx = reinterpret_cast<const u32a*>(row)[(j >> 1) + 1];  // past the last row: the arrays behind G
            }
            gm = ((u & 1) ? e2 >> 22 : (e2 >> 6) & 1023u) - 1u;
            k = (u & 1) ? (e2 >> 16) & 63u : e2 & 63u;
        } else {
            gm = (nx >> 6) - 1u;
            k = nx & 63u;
            nx = row[j + 1];
        }
        asm volatile("" : "+v"(gm));
        W = m + gm;
        const int el = u >> 2;
        if constexpr (P16) {
            const int r = el >> 1;
            const uint32_t nw = __builtin_amdgcn_perm(W, w[r], (el & 1) ? 0x05040100u : 0x03020504u);
            w[r] = own[u & 3] ? nw : w[r];
        } else {
            w[el] = own[u & 3] ? W : w[el];
        }
        if constexpr (FAR) row[j] = (RowT)W;
    }
};

template <typename RowT, bool FAR>
__device__ __forceinline__ int split_min(RowT* row, int n, int woff, int sub) {
    SplitChain<RowT, FAR> ch(row, sub);
    int j0 = 0;
    // whole blocks of 16 steps (no exit inside), then the block that holds label n
    for (; j0 + 16 <= n; j0 += 16) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            uint32_t m = ch.minimum(u, j0 + u);
            if (u == 0) m = j0 == 0 ? (uint32_t)woff : m;
            ch.advance(u, j0 + u, m);
        }
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        uint32_t m = ch.minimum(u, j0 + u);
        if (u == 0) m = j0 == 0 ? (uint32_t)woff : m;
        if (j0 + u == n) return (int)m;
        ch.advance(u, j0 + u, m);
    }
    return 0;  // not reached: n - j0 < 16
}

template <int NTHR, typename RowT>
__device__ __forceinline__ void rank_cost(const CvLds<RowT>& L, int pop, int m, int tid) {
    for (int i = tid; i < pop; i += NTHR) {
        const int q = i / m, base = q * m, il = i - base;
        const int32_t fi = L.cost[i];
        int r = 0;
        for (int p = 0; p < m; ++p) {
            const int32_t fp = L.cost[base + p];
            r += (fp < fi || (fp == fi && p < il)) ? 1 : 0;
        }
        L.ord[base + r] = i;
    }
}

template <typename RowT, int NTHR>
__global__ __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(4))) void cvrp_epoch_kernel(
    CvrpArgs a, const int* __restrict__ order) {
    extern __shared__ __align__(16) uint8_t cv_smem[];
    const int inst = order[blockIdx.x];
    const CvrpDev cd = a.inst[inst];
    const int n = cd.n, cap = cd.cap, pop = cd.pop, S = n + 1;
    const int NP = (n + 3) & ~3, popP = a.popP, tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int GW = cv_row_words(n, sizeof(RowT)) * 4 / (int)sizeof(RowT);  // row stride in entries
    CvLds<RowT> L;
    uint8_t* p = cv_smem;
    L.node = reinterpret_cast<uint2*>(p);
    p += ((S + 1) & ~1) * 8;
    L.G = reinterpret_cast<RowT*>(p);
    p += kCvBatch * GW * sizeof(RowT);
    L.cost = reinterpret_cast<int32_t*>(p);
    L.ord = L.cost + popP;
    L.aux = L.ord + popP;
    L.cur = L.aux + popP;
    L.info = L.cur + popP;
    p += 4 * popP * 4 + kCvBatch * 4;
    L.T = p;
    const int TN = popP * NP;
    const Rng rng{a.seed_lo, a.seed_hi, (uint32_t)inst};
    const int m = pop / (a.n_islands > 0 ? a.n_islands : 1);

    for (int e = tid; e < S; e += NTHR) {
        const uint32_t c = a.xy[cd.xy_off + e];
        L.node[e] = make_uint2(c, (uint32_t)nint_xy(0u, c) | ((uint32_t)a.dem[cd.dem_off + e] << 8));
    }
    for (int i = tid; i < popP; i += NTHR) L.cur[i] = 0;
    uint8_t* tg = a.tours + cd.tour_off;
    if (!a.init) {
        for (int e = tid; e < pop * n; e += NTHR) {
            const int i = e / n, k = e - i * n;
            L.T[i * NP + k] = tg[e];
        }
        for (int i = tid; i < pop; i += NTHR) L.cost[i] = a.cost[cd.cost_off + i];
    } else {
        for (int i = tid; i < pop; i += NTHR) {
            uint8_t* tour = L.T + i * NP;
            for (int k = 0; k < n; ++k) tour[k] = (uint8_t)(k + 1);
            U4 blk{0u, 0u, 0u, 0u};
            for (int k = n - 1; k >= 1; --k) {
                const int w = n - 1 - k;
                if ((w & 3) == 0) blk = rng.block(0u, P_CV_INIT, (uint32_t)i, 0u, (uint32_t)(w >> 2));
                const int j = (int)(pick(blk, (uint32_t)(w & 3)) % (uint32_t)(k + 1));
                const uint8_t tmp = tour[k];
                tour[k] = tour[j];
                tour[j] = tmp;
            }
        }
    }
    __syncthreads();

    // the split of the pass's rows, four lanes each; cost and selection
    auto split_pass = [&](int i0, int cnt, bool init) {
        if (tid < 4 * kCvBatch) {
            const int q = tid >> 2, sub = tid & 3;
            if (16 * wave >= cnt) return;
            const int qe = q < cnt ? q : 16 * wave;  // idle quads repeat their wave's first row
            RowT* row = L.G + qe * GW;
            const int inf = L.info[qe];
            const int mw = __ballot(inf < 0) ? split_min<RowT, true>(row, n, cd.woff, sub)
                                             : split_min<RowT, false>(row, n, cd.woff, sub);
            const int32_t V = (inf & 0x7FFFFFFF) + mw - cd.woff;
            if (q < cnt && sub == 0 && (init || V <= L.cost[i0 + q])) {
                L.cost[i0 + q] = V;
                if (!init) L.cur[i0 + q] |= 2;
            }
        }
    };

    if (a.init) {
        for (int i0 = 0; i0 < pop; i0 += kCvBatch) {
            const int cnt = pop - i0 < kCvBatch ? pop - i0 : kCvBatch;
            for (int q = wave; q < cnt; q += NTHR / 64) {
                const uint8_t* const t[1] = {L.T + (i0 + q) * NP};
                RowT* const row[1] = {L.G + q * GW};
                int32_t* const info[1] = {L.info + q};
                split_data<4, 1>(t, row, info, L.node, n, cap, lane);
            }
            __syncthreads();
            split_pass(i0, cnt, true);
            __syncthreads();
        }
    }

    const float thr1 = a.p_swap, thr2 = a.p_swap + a.p_2opt;
    for (int gen = a.g0 + 1; gen <= a.g1; ++gen) {
        for (int i0 = 0; i0 < pop; i0 += kCvBatch) {
            const int cnt = pop - i0 < kCvBatch ? pop - i0 : kCvBatch;
            // lane l draws for the wave's l-th individual of the pass (row wave + 8 l)
            const int ql = wave + (NTHR / 64) * (lane & 7);
            const int i = i0 + (ql < cnt ? ql : 0);
            const int il = i % m, base = i - il;
            const U4 b0 = rng.block((uint32_t)gen, P_CV_GEN, (uint32_t)i, 0u, 0u);
            const U4 b1 = rng.block((uint32_t)gen, P_CV_GEN, (uint32_t)i, 1u, 0u);
            int r = (int)(b0.x % (uint32_t)(m - 1));
            if (r >= il) r += 1;
            int ca = (int)(b0.y % (uint32_t)n), cb = (int)(b0.z % (uint32_t)n);
            if (ca > cb) { const int t = ca; ca = cb; cb = t; }
            const float u = uniform01(b0.w);
            const int mut = (u < thr1) ? 1 : ((u < thr2) ? 2 : 0);
            const int mc = (int)(b1.x % (uint32_t)n), md = (int)(b1.y % (uint32_t)n);
            const int c1 = L.cur[i] & 1, c2 = L.cur[base + r] & 1;
            const int cuts = ca | (cb << 8) | (mc << 16) | (md << 24);  // n <= 255
            const int rest = (base + r) | (mut << 10) | (c1 << 12) | (c2 << 13);
            // rows l .. l + NI - 1 of the wave; a row past the pass repeats the one before
            auto breed = [&](auto nc, auto ni, int l) {
                constexpr int NC = decltype(nc)::value, NI = decltype(ni)::value;
                Breed bd[NI];
                uint8_t* rows[NI];
                const uint8_t* t[NI];
                RowT* row[NI];
                int32_t* info[NI];
#pragma unroll
                for (int e = 0; e < NI; ++e) {
                    const int le = wave + (NTHR / 64) * (l + e) < cnt ? l + e : l;
                    const int q = wave + (NTHR / 64) * le;
                    const uint32_t v = (uint32_t)__builtin_amdgcn_readlane(cuts, le);
                    const uint32_t w = (uint32_t)__builtin_amdgcn_readlane(rest, le);
                    const int self = (w >> 12) & 1, mt = (w >> 10) & 3;
                    const int x = (v >> 16) & 255, y = v >> 24, lo = x < y ? x : y, hi = x < y ? y : x;
                    bd[e].p1 = L.T + self * TN + (i0 + q) * NP;
                    bd[e].p2 = L.T + (int)((w >> 13) & 1u) * TN + (int)(w & 1023u) * NP;
                    bd[e].child = L.T + (self ^ 1) * TN + (i0 + q) * NP;
                    bd[e].a = v & 255;
                    bd[e].b = (v >> 8) & 255;
                    // 1: lo and hi exchanged, 2: lo .. hi reversed, 0: nothing (no position is that far)
                    bd[e].lo = mt ? lo : 1 << 20;
                    bd[e].span = mt == 2 ? hi - lo : 0;
                    bd[e].hi = mt ? hi : -1;
                    bd[e].sum = lo + hi;
                    row[e] = L.G + q * GW;
                    rows[e] = reinterpret_cast<uint8_t*>(row[e]);
                    t[e] = bd[e].child;
                    info[e] = L.info + q;
                }
                make_children<NC, NI>(bd, rows, n, lane);
                split_data<NC, NI>(t, row, info, L.node, n, cap, lane);
            };
            using std::integral_constant;
            for (int l = 0; wave + (NTHR / 64) * l < cnt; l += n <= 128 ? 2 : 1) {
                if (n <= 64) breed(integral_constant<int, 1>{}, integral_constant<int, 2>{}, l);
                else if (n <= 128) breed(integral_constant<int, 2>{}, integral_constant<int, 2>{}, l);
                else if (n <= 192) breed(integral_constant<int, 3>{}, integral_constant<int, 1>{}, l);
                else breed(integral_constant<int, 4>{}, integral_constant<int, 1>{}, l);
            }
            __syncthreads();
            split_pass(i0, cnt, false);
            __syncthreads();
        }
        // accepted children become the individuals once every child of the generation is made
        for (int i = tid; i < pop; i += NTHR) {
            const int c = L.cur[i];
            L.cur[i] = (c ^ (c >> 1)) & 1;
        }
        __syncthreads();
        const int nis = a.n_islands, kk = a.migrate_count;
        if (nis > 1 && a.migrate_interval > 0 && kk > 0 && gen % a.migrate_interval == 0) {
            rank_cost<NTHR>(L, pop, m, tid);
            __syncthreads();
            for (int e = tid; e < nis * kk; e += NTHR) {
                const int q = e / kk, j = e - q * kk, pd = (q + 1) % nis;
                const int src = L.ord[q * m + j], dst = L.ord[pd * m + m - kk + j];
                L.aux[e] = (L.cost[src] < L.cost[dst]) ? 1 : 0;
            }
            __syncthreads();
            for (int e = tid; e < nis * kk * (NP / 4); e += NTHR) {
                const int pr = e / (NP / 4), w = e - pr * (NP / 4);
                if (L.aux[pr]) {
                    const int q = pr / kk, j = pr - q * kk, pd = (q + 1) % nis;
                    const int src = L.ord[q * m + j], dst = L.ord[pd * m + m - kk + j];
                    reinterpret_cast<uint32_t*>(L.T + L.cur[dst] * TN + dst * NP)[w] =
                        reinterpret_cast<const uint32_t*>(L.T + L.cur[src] * TN + src * NP)[w];
                }
            }
            for (int e = tid; e < nis * kk; e += NTHR) {
                if (L.aux[e]) {
                    const int q = e / kk, j = e - q * kk, pd = (q + 1) % nis;
                    const int src = L.ord[q * m + j], dst = L.ord[pd * m + m - kk + j];
                    L.cost[dst] = L.cost[src];
                }
            }
            __syncthreads();
        }
    }
    for (int e = tid; e < pop * n; e += NTHR) {
        const int i = e / n, k = e - i * n;
        tg[e] = L.T[L.cur[i] * TN + i * NP + k];
    }
    for (int i = tid; i < pop; i += NTHR) a.cost[cd.cost_off + i] = L.cost[i];
}

// Best individual of every instance (the first of the smallest cost), one wave each: its cost
// and its tour (rows of `stride` bytes), written straight into pinned host memory.
__global__ __launch_bounds__(64) void cvrp_best_kernel(const CvrpDev* __restrict__ inst, const int32_t* __restrict__ cost,
                                                       const uint8_t* __restrict__ tours, int stride,
                                                       int32_t* __restrict__ out_cost, uint8_t* __restrict__ out_tour) {
    const int t = blockIdx.x, lane = threadIdx.x;
    const CvrpDev cd = inst[t];
    int32_t bc = 0x7FFFFFFF;
    int bi = 0;
    for (int i = lane; i < cd.pop; i += 64) {
        const int32_t c = cost[cd.cost_off + i];
        if (c < bc) {
            bc = c;
            bi = i;
        }
    }
#pragma unroll
    for (int w = 32; w >= 1; w >>= 1) {
        const int32_t oc = __shfl_xor(bc, w);
        const int oi = __shfl_xor(bi, w);
        if (oc < bc || (oc == bc && oi < bi)) {
            bc = oc;
            bi = oi;
        }
    }
    if (lane == 0) out_cost[t] = bc;
    const uint8_t* src = tours + cd.tour_off + (int64_t)bi * cd.n;
    uint8_t* dst = out_tour + (int64_t)t * stride;
    for (int k = 4 * lane; k < cd.n; k += 256) {  // stride is a multiple of 4
        uint32_t v = 0;
        for (int b = 0; b < 4; ++b) v |= (uint32_t)(k + b < cd.n ? src[k + b] : 0) << (8 * b);
        *reinterpret_cast<uint32_t*>(dst + k) = v;
    }
}

}  // namespace emtf

extern "C" int emtf_cvrp_launch_best(const emtf::CvrpDev* inst, int n_inst, const int32_t* cost, const uint8_t* tours,
                                     int stride, int32_t* out_cost, uint8_t* out_tour, hipStream_t stream) {
    hipLaunchKernelGGL(emtf::cvrp_best_kernel, dim3(n_inst), dim3(64), 0, stream, inst, cost, tours, stride, out_cost,
                       out_tour);
    return (int)hipGetLastError();
}

extern "C" int emtf_cvrp_lds_bytes(int n, int popP, int entry_bytes) {
    return emtf::cvrp_lds_bytes(n, popP, entry_bytes);
}

template <typename RowT, int NTHR>
static hipError_t launch_epoch(const emtf::CvrpArgs& a, const int* order, int n, int lds_bytes, hipStream_t stream) {
    static bool lds_ok = false;
    auto k = &emtf::cvrp_epoch_kernel<RowT, NTHR>;
    if (!lds_ok) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        lds_ok = true;
    }
    hipLaunchKernelGGL(k, dim3(n), dim3(NTHR), lds_bytes, stream, a, order);
    return hipGetLastError();
}

// entry_bytes 2: W + woff in 16 bits (the host checks that every instance's W + woff range
// fits); else W in 32 bits.  Sixteen waves an instance up to one instance a CU (the registers of
// sixteen waves fill it), eight beyond.  100 generations, 50 to 200 customers, pop 128: 16 / 256
// instances 6.21 / 6.33 ms with eight waves, 5.07 / 5.21 with sixteen; 512 instances 6.55 and 7.20.
extern "C" int emtf_cvrp_launch(const emtf::CvrpArgs* args, const int* order, int n_inst, int lds_bytes, int entry_bytes,
                                hipStream_t stream) {
    constexpr int kCus = 256;
    const bool wide = args->n_inst <= kCus;
    auto* const fn = entry_bytes == 2 ? (wide ? &launch_epoch<uint16_t, 2 * emtf::kCvThreads> : &launch_epoch<uint16_t, emtf::kCvThreads>)
                                      : (wide ? &launch_epoch<uint32_t, 2 * emtf::kCvThreads> : &launch_epoch<uint32_t, emtf::kCvThreads>);
    return (int)fn(*args, order, n_inst, lds_bytes, stream);
}
