// island.hip -- the island-model evolutionary-multitasking kernel for gfx950.
//
// One workgroup (4 wave64s) owns one task for one epoch of generations.  The
// task's population, its transform matrix and its per-dimension tables live in
// LDS for the whole epoch; HBM is touched only to load and store the state at
// the epoch boundaries and for the elite mailbox that carries inter-task
// transfer.  Per generation and per 32-individual tile a wave
//   1. draws its Philox numbers in registers (no RNG state in memory),
//   2. gathers parent/mate rows from LDS and forms the trial vectors,
//   3. computes z = Q (u - o) with v_mfma_f32_32x32x2_f32: B = the trial tile
//      (one individual per column, one gene parity per lane half), A = Q,
//      so each lane ends up holding 16 rows of z for its own individual,
//   4. evaluates the objective on those rows and combines the two lane halves
//      with one cross-half shuffle,
//   5. applies the greedy one-to-one selection in LDS.
//
// Reference operators restated (file:line of proposed model/):
//   GeneticOpera SG-EMTF.cu:1289-1426 / SG-EMTF_DE.cu:1241-1390 (the island loop),
//   CrossOver/Mutation/Selection SG-EMTF_DE.cu:474-705, SG-EMTF.cu:548-831,
//   evaluation SG-EMTF_DE.cu:834-1069, IslandMigration SG-EMTF_DE.cu:1093-1170,
//   SharedToGlobal/SelectFromBlocks SG-EMTF.cu:856-896,1220-1260,
//   knowledgeTransfer SG-EMTF.cu:1514-1591, pop_init SG-EMTF.cu:146-159.
//
// LDS layout of a row (individual i, or row j of Q): the even genes
// 0,2,4,.. in slots [0, HS) and the odd genes in [HS, 2 HS), HS = 4 KB, so a
// lane half streams its parity with 16-byte loads; RS = 2 HS + 4 is the row
// stride.  Slots past the task's dimension hold zeros, which makes every MFMA
// step and every gene block unconditional: padded steps add +0 products.
#include <hip/hip_runtime.h>
#include "emtf_eval.h"
#include "emtf_math.h"
#include "emtf_types.h"

namespace emtf {

constexpr int kThreads = 256;

// Row geometry fixed at compile time: KB blocks of 4 genes per parity half.
template <int KB>
struct Shape {
    static constexpr int HS = 4 * KB;          // slots per parity half
    static constexpr int RS = 2 * HS + 4;      // LDS row stride (floats)
    static constexpr int NT = (KB + 3) / 4;    // 32-row output tiles (dims <= 32 NT)
};

// The gene block from which a build leaves out those that lie past the dimension (0: none):
// about the middle of the dimensions that it takes (the next smaller build takes those up to its
// own 8 KB).  Each skip is a branch, before which the loads of its block are not issued: at D = 37
// (KB = 7, DE, 1024 tasks) an epoch of 20 generations went from 0.301 to 0.266 ms, at D = 50 from
// 0.316 to 0.318 (GA 0.730 to 0.665, 0.851 to 0.863).
template <int KB>
constexpr int kSkipBlock = KB == 4 ? 3 : (KB == 7 ? 5 : (KB == 12 ? 10 : (KB == 16 ? 14 : 0)));

// Q in the matrix instructions' operand order (an image built on the device when a batch is
// created): 256 floats per gene block and row tile, lane l's four the genes of the block in half
// l >> 5 of row 32 jt + (l & 31), zero past the dimension.  A wave's read is 1 KB of consecutive
// bytes -- from L2 where a row-major matrix costs 64 lines of 16 bytes each, from LDS without a
// bank conflict or the rows' padding.
__device__ __forceinline__ float4 q_op(const float* q, int nt, int sb, int jt) {
    const float* p = q + 256 * (sb * nt + jt);
    return make_float4(p[0], p[1], p[2], p[3]);
}

// LDS-kernel builds that read Q's image (of kQTiles row tiles) from L2, a block ahead of its
// use: from KB = 12 on the rows and Q together leave room for one workgroup a CU, a wave per
// SIMD that issues an instruction each 5.7 cycles; the rows alone for two.  D = 100, pop 128, an
// epoch of 20 generations: 1024 sphere tasks 1.145 to 0.826 ms, Weierstrass 3.66 to 1.77; 256
// tasks (one workgroup a CU either way) 0.312 to 0.281 and 0.945 to 0.719.
template <int KB>
constexpr bool kQGlobal = KB >= 12;
constexpr int kQTiles = 4;

struct Geo {
    int D, Dh, pop, popP, ntiles, m;
    FastMod modD, modM;  // jrand = w mod D, island-local index = w mod m
};

struct Lds {
    float* X;    // popP x RS
    float* Q;    // 32 NT x RS
    float* o;    // RS
    float* tab;  // 32 NT
    float* fit;  // popP
    float* ftmp; // popP
    int* ord;    // popP
    int* aux;    // popP
};

__host__ __device__ inline int lds_floats_kb(int pop, int kb) {
    const int RS = 8 * kb + 4, NT = (kb + 3) / 4, popP = (pop + 31) & ~31;
    return popP * RS + 32 * NT * RS + RS + 32 * NT + 4 * popP;
}

// What the epoch kernel allocates: the same, without Q where it reads the image.
__host__ __device__ inline int epoch_lds_floats(int pop, int kb) {
    return lds_floats_kb(pop, kb) - (kb >= 12 ? 32 * ((kb + 3) / 4) * (8 * kb + 4) : 0);
}

// v clamped to [lo, hi] (hi if v > hi, else lo if v < lo, else v: a NaN stays NaN), as
// two selects.
__device__ __forceinline__ float clampf(float v, float lo, float hi) {
    const float t = v < lo ? lo : v;
    return v > hi ? hi : t;
}

// The box clamp of a trial gene as one median: equal to clampf for every
// non-NaN value (trial genes are always finite) except a signed-zero tie with a bound
// of zero, which the engine never produces (a -0 gene needs a -0 parent, and the
// initial population of a box starting at 0 holds none).
__device__ __forceinline__ float clamp_box(float v, float lo, float hi) {
    return __builtin_amdgcn_fmed3f(v, lo, hi);
}

// A replayed epoch (hipGraph) starts at the device generation counter: its launch
// arguments were frozen when the graph was captured, the counter advances every replay.
__device__ __forceinline__ void rebase_epoch(EpochArgs& a) {
    if (a.gen_dev) {
        const int g0 = *a.gen_dev;
        a.g1 = g0 + (a.g1 - a.g0);
        a.g0 = g0;
    }
}

// Online admission: a task takes part in the epochs that lie inside its life and is
// initialised by the launch at its admission (every task of a handle created without
// online admission: gen_base 0, gen_end INT32_MAX).
__device__ __forceinline__ bool runs_epoch(const EpochArgs& a, const TaskDev& td) {
    return a.init ? td.gen_base == a.g0 : (td.gen_base <= a.g0 && a.g1 <= td.gen_end);
}

// Whether the task receives elites at the start of this epoch: a transfer boundary that
// is not its own start, with another donor to draw.
// (g0: the epoch's first generation, a.g0 but for the persistent schedule's items)
__device__ __forceinline__ bool transfer_now(const EpochArgs& a, const TaskDev& td, int g0) {
    const int TI = a.p.transfer_interval;
    if (a.init || TI <= 0 || a.p.transfer_count <= 0 || g0 % TI != 0 || g0 <= td.gen_base) return false;
    return a.donors ? *a.n_donors > 1 : a.n_tasks > 1;
}
__device__ __forceinline__ bool transfer_now(const EpochArgs& a, const TaskDev& td) { return transfer_now(a, td, a.g0); }

// The donor of task `task` at a transfer event: the k-th of the other donors in ascending
// id order, k = w mod (n - 1) -- every task of the handle, or the online donor list.
__device__ __forceinline__ int pick_donor(const EpochArgs& a, int task, uint32_t w) {
    if (!a.donors) {
        const int dn = (int)(w % (uint32_t)(a.n_tasks - 1));
        return dn >= task ? dn + 1 : dn;
    }
    const int n = *a.n_donors;
    const int k = (int)(w % (uint32_t)(n - 1));
    int lo = 0, hi = n - 1;  // the task's own position in the list (it is a donor itself)
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a.donors[mid] < task) lo = mid + 1;
        else hi = mid;
    }
    return a.donors[k + (k >= lo ? 1 : 0)];
}

// z = Q (x - o) for the 32 individuals of a tile (x: the lane's parity half)
// followed by the objective.  One MFMA k-step per gene pair (2 p, 2 p + 1), p < Dh:
// the steps past the dimension would add q * 0 products of the zero padding, which
// leave the accumulator unchanged (it is never -0), so they are skipped (a uniform
// branch, taken only in the last blocks).
template <int KB, int FUNC>
__device__ __forceinline__ float evaluate_tile(const float (&x)[4 * KB], const Geo& g, const Lds& L, int col, int h) {
    using S = Shape<KB>;
    constexpr int NT = S::NT;
    f16v acc[NT];
#pragma unroll
    for (int jt = 0; jt < NT; ++jt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[jt][r] = 0.0f;
    const float* qrow = kQGlobal<KB> ? L.Q + 4 * (32 * h + col) : L.Q + col * S::RS + h * S::HS;
    const float* orow = L.o + h * S::HS;
#pragma unroll
    for (int sb = 0; sb < KB; ++sb) {
        float4 q[NT];
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
            q[jt] = kQGlobal<KB> ? q_op(qrow, kQTiles, sb, jt) : lds4(qrow + 32 * jt * S::RS + 4 * sb);
        const float4 o4 = lds4(orow + 4 * sb);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (sb < KB - 1 || 4 * sb + e < g.Dh) {
                const float w = x[4 * sb + e] - f4(o4, e);
#pragma unroll
                for (int jt = 0; jt < NT; ++jt)
                    acc[jt] = __builtin_amdgcn_mfma_f32_32x32x2f32(f4(q[jt], e), w, acc[jt], 0, 0, 0);
            }
        }
    }
    return objective<NT, FUNC>(acc, g.D, L.tab, h);
}

// ---------------------------------------------------------------------------
// Trial vectors
// ---------------------------------------------------------------------------
struct IdxStream {
    uint32_t w0, w1, w2, w3;
    int wi, wn, blk;
};

__device__ __forceinline__ bool idx_next(IdxStream& st, const Rng& rng, uint32_t gen, uint32_t index, uint32_t& out) {
    if (st.wi == st.wn) {
        if (st.blk == 3) return false;
        st.blk += 1;
        const U4 b = rng.block(gen, P_DE_IDX, index, 0u, (uint32_t)st.blk);
        st.w0 = b.x; st.w1 = b.y; st.w2 = b.z; st.w3 = b.w;
        st.wn = 4;
        st.wi = 0;
    }
    out = st.wi == 0 ? st.w0 : (st.wi == 1 ? st.w1 : (st.wi == 2 ? st.w2 : st.w3));
    st.wi += 1;
    return true;
}

// Rejection draw of an island-local index outside excl[0..nex) (reference
// CrossOver, SG-EMTF_DE.cu:559-573: redraw curand()%n while it collides).
__device__ __forceinline__ int draw_excl(IdxStream& st, const Rng& rng, uint32_t gen, uint32_t index, int m,
                                         const int* excl, int nex) {
    int distinct = 0;
    for (int a = 0; a < nex; ++a) {
        int dup = 0;
        for (int b = 0; b < a; ++b) dup |= (excl[b] == excl[a]);
        distinct += !dup;
    }
    uint32_t w;
    while (idx_next(st, rng, gen, index, w)) {
        const int r = (int)(w % (uint32_t)m);
        int bad = 0;
        if (distinct < m)
            for (int a = 0; a < nex; ++a) bad |= (excl[a] == r);
        if (!bad) return r;
    }
    for (int r = 0; r < m; ++r) {
        int bad = 0;
        for (int a = 0; a < nex; ++a) bad |= (excl[a] == r);
        if (!bad) return r;
    }
    return 0;
}

// DE mates of individual ie (island-local indices) and jrand: the first three words
// of its index stream usually give admissible mates (no rejection); otherwise the
// sequential rejection draw is replayed, which then consumes more words.
struct DeMates {
    int r1, r2, r3, jrand;
};

__device__ __forceinline__ DeMates de_mates(const EpochArgs& a, const Geo& g, const Rng& rng, int gen, int ie) {
    const int m = g.m, il = (int)g.modM.mod((uint32_t)ie);
    const bool rand1 = (a.p.algo == A_DE_RAND_1_BIN);
    const U4 b0 = rng.block((uint32_t)gen, P_DE_IDX, (uint32_t)ie, 0u, 0u);
    DeMates r;
    r.jrand = (int)g.modD.mod(b0.w);
    r.r1 = (int)g.modM.mod(b0.x);
    r.r2 = (int)g.modM.mod(b0.y);
    r.r3 = (int)g.modM.mod(b0.z);
    const bool ok = rand1 ? (m >= 4 && r.r1 != il && r.r2 != il && r.r2 != r.r1 && r.r3 != il && r.r3 != r.r1 && r.r3 != r.r2)
                          : (m >= 3 && r.r2 != r.r1 && r.r3 != r.r1 && r.r3 != r.r2);
    bool replay = !ok;
    if (!ok && m >= 4) {
        // the rejection draws over the first seven words of the stream (block 0's x, y,
        // z, then block 1) in straight-line code: each word is taken by the first mate
        // still missing unless it collides with an excluded index; with m >= 4 every draw
        // has an admissible value, so this is the sequential rejection draw whenever
        // seven words suffice (a lane needing more replays it below)
        const U4 b1 = rng.block((uint32_t)gen, P_DE_IDX, (uint32_t)ie, 0u, 1u);
        const uint32_t w[7] = {b0.x, b0.y, b0.z, b1.x, b1.y, b1.z, b1.w};
        int got = 0, q1 = 0, q2 = 0, q3 = 0;
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            const int v = (k == 0) ? r.r1 : ((k == 1) ? r.r2 : ((k == 2) ? r.r3 : (int)g.modM.mod(w[k])));
            const bool bad = (rand1 && v == il) || (got >= 1 && v == q1) || (got >= 2 && v == q2);
            const bool take = !bad && got < 3;
            q1 = (take && got == 0) ? v : q1;
            q2 = (take && got == 1) ? v : q2;
            q3 = (take && got == 2) ? v : q3;
            got += take ? 1 : 0;
        }
        r.r1 = q1;
        r.r2 = q2;
        r.r3 = q3;
        replay = got < 3;
    }
    if (replay) {
        IdxStream st{b0.x, b0.y, b0.z, 0u, 0, 3, 0};
        int ex[3];
        int nex = 0;
        if (rand1) ex[nex++] = il;
        r.r1 = draw_excl(st, rng, (uint32_t)gen, (uint32_t)ie, m, ex, nex);
        ex[nex++] = r.r1;
        r.r2 = draw_excl(st, rng, (uint32_t)gen, (uint32_t)ie, m, ex, nex);
        ex[nex++] = r.r2;
        r.r3 = draw_excl(st, rng, (uint32_t)gen, (uint32_t)ie, m, ex, nex);
    }
    return r;
}

// The two halves of a wave hold the same individuals, and draws depend on the generation
// number only: at the first of two generations the lower half draws that generation's mates
// and the upper half the next one's, which `next` carries over (m: island-local mates, 10
// bits each, j: jrand).
struct MateCache {
    uint32_t m, j;
};

__device__ __forceinline__ DeMates de_mates2(const EpochArgs& a, const Geo& g, const Rng& rng, int gen, int ie, int h,
                                             bool first, MateCache& next) {
    uint32_t m, j;
    if (first) {
        const DeMates r = de_mates(a, g, rng, gen + h, ie);
        m = (uint32_t)(r.r1 | (r.r2 << 10) | (r.r3 << 20));
        j = (uint32_t)r.jrand;
        typedef unsigned u2 __attribute__((ext_vector_type(2)));
        const u2 sm = __builtin_amdgcn_permlane32_swap(m, m, false, false);
        const u2 sj = __builtin_amdgcn_permlane32_swap(j, j, false, false);
        m = sm.x;
        j = sj.x;
        next.m = sm.y;
        next.j = sj.y;
    } else {
        m = next.m;
        j = next.j;
    }
    return DeMates{(int)(m & 1023u), (int)((m >> 10) & 1023u), (int)(m >> 20), (int)j};
}

// Genes 2 s + h, s = 4 sb .. 4 sb + 3, of a DE/x/1/bin trial: mutant vb + F (v2 - v3)
// clamped to the box, binomial crossover with the parent vi (16-bit uniforms from
// block cb: two gene blocks per Philox block).  Slots past the dimension are left as
// computed (finite, inside the box): every reader of a row takes its first D genes only,
// and the rotation meets them only in k-steps whose Q entries are zero.
//
// Operand rule of the vector unit (measured): a float add, multiply or fma takes 2 cycles on
// vector registers and literals, 4 with a scalar register, and compares, selects, shifts
// and min / max take 4 whatever they read.  So F and the box come in vector registers, the
// box clamp is one median, and the 16-bit uniforms are compared where they lie in their word
// (the upper half: the whole word against a threshold shifted up) instead of extracted.  With
// the mates above and four blocks' draws at a time, an epoch of 20 generations of 1024 tasks
// (D = 50, pop 128): sphere 0.356 to 0.314 ms, Ackley 0.396 to 0.354, all eight 0.518 to 0.454.
struct DeConst {
    float F, lo, hi;
    uint32_t thi, tlo;  // keep the parent iff (word & ~1) >= thi | its lower half >= tlo
    int jr;             // jrand - h
};

__device__ __forceinline__ DeConst de_const(const EpochArgs& a, const TaskDev& td) {
    DeConst c;
    c.F = a.p.F;
    c.lo = td.lo;
    c.hi = td.hi;
    asm volatile("" : "+v"(c.F), "+v"(c.lo), "+v"(c.hi));
    // upper half >= t  <=>  word with its lowest bit cleared >= t 2^16 (t = 2^16: 2^32 - 1, never)
    c.tlo = a.p.cr_threshold;
    c.thi = c.tlo < 65536u ? c.tlo << 16 : 0xFFFFFFFFu;
    c.jr = 0;
    return c;
}

// Gene e of the block (slot s = 4 sb + e).
__device__ __forceinline__ float de_gene(const DeConst& c, float vb, float v2, float v3, float vi, const U4& cb, int sb,
                                         int e) {
    // gene d = 2 s + h: the test d == jrand is made on 2 s against the lane's jrand - h,
    // so no per-gene index is held in a register
    const int s2 = 2 * (4 * sb + e);
    const float diff = v2 - v3;
    const float sc = c.F * diff;
    float v = vb + sc;
    v = clamp_box(v, c.lo, c.hi);
    const uint32_t w = pick(cb, (uint32_t)(((sb & 1) << 1) | (e >> 1)));
    const bool keep = (e & 1) ? (w & 0xFFFFu) >= c.tlo : (w & ~1u) >= c.thi;
    return (keep & (s2 != c.jr)) ? vi : v;
}

__device__ __forceinline__ void de_block(float (&t)[4], const float4& vb, const float4& v2, const float4& v3,
                                         const float4& vi, const U4& cb, int sb, const DeConst& c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = de_gene(c, f4(vb, e), f4(v2, e), f4(v3, e), f4(vi, e), cb, sb, e);
}

// Genes 2 s + h, s = 4 sb .. 4 sb + 3, of a GA child: SBX of parents va, vb
// (spread sign by the child's parity in its pair) then polynomial mutation,
// each clamped to the box, zero past the dimension.
struct GaConst {
    float lo, hi, rng, ec, em1, em, pm;
    float inv;         // 1 / rng
    float at1, at2;    // 0^em1, 0^em
    bool plain;        // box, range and exponents far from the exponent range's ends (see ga_const)
};

// Gene of a GA child, general: any parameters, any box.  sbw, r, uw: the gene's draws.
__device__ __forceinline__ float ga_gene(float va, float vb, uint32_t sbw, uint32_t rw, uint32_t uw, bool odd,
                                         const GaConst& c0) {
    const float lo = c0.lo, hi = c0.hi, rng_ = c0.rng;
    const float p = uniform_open(sbw);
    const float tv = (p <= 0.5f) ? (2.0f * p) : (0.5f / (1.0f - p));
    float beta = pow_f(tv, c0.ec);
    if (odd) beta = -beta;
    const float t1 = 1.0f + beta;
    const float t2 = t1 * va;
    const float t3 = 1.0f - beta;
    const float t4 = t3 * vb;
    const float t5 = t2 + t4;
    float c = 0.5f * t5;
    c = clamp_box(c, lo, hi);
    const float r = uniform01(rw);
    if (r < c0.pm) {
        const float u = uniform01(uw);
        float delta = 1.0f, iv1, iv2, dl;
        const float num = c - lo;
        dl = num / rng_;
        iv1 = 2.0f * u;
        iv2 = 1.0f - iv1;
        if (u > 0.5f) {
            delta = -1.0f;
            const float num2 = hi - c;
            dl = num2 / rng_;
            const float omu = 1.0f - u;
            iv1 = 2.0f * omu;
            const float um = u - 0.5f;
            iv2 = 2.0f * um;
        }
        const float omd = 1.0f - dl;
        const float pw = pow_f(omd, c0.em1);
        const float a2 = iv2 * pw;
        const float a3 = iv1 + a2;
        const float a4 = pow_f(a3, c0.em);
        const float a5 = a4 - 1.0f;
        delta = delta * a5;
        const float step = delta * rng_;
        c = c + step;
        c = clamp_box(c, lo, hi);
    }
    return c;
}

// Genes 2 s + h, s = 4 sb .. 4 sb + 3, of a GA child: SBX of parents va, vb
// (spread sign by the child's parity in its pair) then polynomial mutation,
// each clamped to the box, zero past the dimension.  What bounds it: three powers and two
// quotients per gene.  They are taken by the forms for the arguments these operators
// nearly always have (the same values); a block with a gene outside them is done again by the
// general one, a rolled loop.  An epoch of 20 generations of 1024 tasks (D = 50, pop 128): 1.72 to
// 1.25 ms.
__device__ __forceinline__ void ga_block(float (&t)[4], const float4& va, const float4& vb, const Rng& rng, int gen,
                                         int ie, int sb, int h, bool odd, int D, const GaConst& c0) {
    U4 db[3];  // SBX draws, then the mutation's
    const uint32_t adr = (((uint32_t)h & 0xFFu) << 16) | ((uint32_t)ie & 0xFFFFu);
    const uint32_t w0[3] = {(uint32_t)sb, (uint32_t)(2 * sb), (uint32_t)(2 * sb + 1)};
    const uint32_t w1[3] = {(P_GA_SBX << 24) | adr, (P_GA_PM << 24) | adr, (P_GA_PM << 24) | adr};
    philox_blocks<3>(db, w0, w1, (uint32_t)gen, rng.task, rng.k0, rng.k1);
    const float lo = c0.lo, hi = c0.hi, rng_ = c0.rng;
    const int dlim = D - h;  // gene 2 s + h < D  <=>  2 s < D - h
    bool ok = c0.plain;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        t[e] = 0.0f;
        if (2 * (4 * sb + e) >= D) continue;  // past the dimension in both halves (a uniform branch)
        const float p = uniform_open(pick(db[0], (uint32_t)e));  // (2 k + 1) 2^-24
        // the division's operand is 1 - p where p > 1/2 (exact); both branches in one select
        const float tv = (p <= 0.5f) ? (2.0f * p) : (0.5f * recip24(1.0f - p));
        float beta = pow_mid(tv, c0.ec);  // 2^-23 <= tv <= 2^23
        if (odd) beta = -beta;
        const float t1 = 1.0f + beta;
        const float t2 = t1 * f4(va, e);
        const float t3 = 1.0f - beta;
        const float t4 = t3 * f4(vb, e);
        const float t5 = t2 + t4;
        float c = 0.5f * t5;
        c = clamp_box(c, lo, hi);
        const U4& pb = (e < 2) ? db[1] : db[2];
        const float r = uniform01(pick(pb, (uint32_t)((e & 1) * 2)));
        if (r < c0.pm) {
            const float u = uniform01(pick(pb, (uint32_t)((e & 1) * 2 + 1)));
            const bool up = u > 0.5f;
            const float num = up ? hi - c : c - lo;
            const float dl = quot_by(num, rng_, c0.inv);
            const float omu = 1.0f - u;
            const float um = u - 0.5f;
            const float iv1 = 2.0f * (up ? omu : u);
            const float iv2 = up ? 2.0f * um : 1.0f - iv1;
            const float omd = 1.0f - dl;
            // omd is 0 or at least 2^-25 (dl <= 1); a3 may be subnormal where u = 1
            const float pm = pow_mid(omd, c0.em1);
            const float pw = omd == 0.0f ? c0.at1 : pm;
            const float a2 = iv2 * pw;
            const float a3 = iv1 + a2;
            const float pn = pow_mid(a3, c0.em);
            const float a4 = a3 == 0.0f ? c0.at2 : pn;
            ok = ok & ((a3 == 0.0f) | (__float_as_uint(a3) - 0x00800000u < 0x7F000000u));
            const float a5 = a4 - 1.0f;
            const float delta = up ? -a5 : a5;
            const float step = delta * rng_;
            c = c + step;
            c = clamp_box(c, lo, hi);
        }
        t[e] = c;
    }
    if (!ok) {
#pragma unroll 1
        for (int e = 0; e < 4; ++e) {
            const U4& pb = (e < 2) ? db[1] : db[2];
            const float c = ga_gene(f4(va, e), f4(vb, e), pick(db[0], (uint32_t)e),
                                    pick(pb, (uint32_t)((e & 1) * 2)), pick(pb, (uint32_t)((e & 1) * 2 + 1)), odd, c0);
#pragma unroll
            for (int f = 0; f < 4; ++f) t[f] = e == f ? c : t[f];
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = (8 * sb + 8 <= D || 2 * (4 * sb + e) < dlim) ? t[e] : 0.0f;
}

__device__ __forceinline__ GaConst ga_const(const EpochArgs& a, const TaskDev& td) {
    GaConst c;
    c.lo = td.lo;
    c.hi = td.hi;
    c.rng = td.hi - td.lo;
    c.ec = 1.0f / (a.p.eta_c + 1.0f);
    c.em1 = a.p.eta_m + 1.0f;
    c.em = 1.0f / c.em1;
    c.pm = a.p.pm;
    c.inv = 1.0f / c.rng;
    auto zero_pow = [](float y) { return y > 0.0f ? 0.0f : (y == 0.0f ? 1.0f : __builtin_inff()); };
    c.at1 = zero_pow(c.em1);
    c.at2 = zero_pow(c.em);
    // quot_by's operands: with both bounds at least 2^-30 a nonzero distance to one is at
    // least 2^-55, so numerator, range, quotient and remainders are normal
    const float b0 = __builtin_fabsf(c.lo), b1 = __builtin_fabsf(c.hi);
    c.plain = b0 >= 9.31322575e-10f && b1 >= 9.31322575e-10f && b0 <= 1.0e15f && b1 <= 1.0e15f &&
              c.rng >= 9.31322575e-10f && __builtin_fabsf(c.ec) <= 1000.0f && __builtin_fabsf(c.em1) <= 1000.0f &&
              __builtin_fabsf(c.em) <= 1000.0f;
    // in vector registers: as scalars they (and what is live beside them) are spilled and come
    // back as lane reads, 14 of a gene's 200 instructions (1024 sphere tasks, D = 50, pop 128:
    // 0.93 to 0.85 ms an epoch)
    asm volatile("" : "+v"(c.lo), "+v"(c.hi), "+v"(c.rng), "+v"(c.inv), "+v"(c.ec), "+v"(c.em1), "+v"(c.em), "+v"(c.pm));
    return c;
}

// The lane's trial half-row, block by block, each block's four genes fed straight into
// the MFMA k-steps of z = Q (x - o), so no lane holds a whole row (on gfx950 the FP32
// MFMA and the VALU share the SIMD's issue: measured, neither overlaps the other, so the
// interleaving saves registers, not time).  The same genes, k order and accumulators as
// generating the whole row first and then evaluating it.
// The trial genes are left in tr (for the selection copy); returns f of the trial.
template <int KB, int FUNC, int ALGO>
__device__ __forceinline__ float trial_eval(float (&tr)[4 * KB], const EpochArgs& a, const TaskDev& td, const Geo& g,
                                            const Lds& L, const Rng& rng, int gen, int ie, int col, int h_in,
                                            bool pair, bool first, MateCache& next) {
    using S = Shape<KB>;
    // the lane's half index is made opaque here: otherwise the compiler hoists every
    // mask and address derived from it out of the generation loop, where the lane masks
    // outgrow the scalar registers and come back from spill slots each generation
    int h = h_in;
    asm volatile("" : "+v"(h));
    constexpr int NT = S::NT;
    const int off = h * S::HS;
    const int il = (int)g.modM.mod((uint32_t)ie), base = ie - il;
    f16v acc[NT];
#pragma unroll
    for (int jt = 0; jt < NT; ++jt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[jt][r] = 0.0f;
    const float* qrow = kQGlobal<KB> ? L.Q + 4 * (32 * h + col) : L.Q + col * S::RS + off;
    const float* orow = L.o + off;
    float4 qn[NT];  // the next block's, loaded a block ahead from L2
    if constexpr (kQGlobal<KB>) {
#pragma unroll
        for (int jt = 0; jt < NT; ++jt) qn[jt] = q_op(qrow, kQTiles, 0, jt);
    }
    // GA: the pair's mates and constants; DE: the three mates and jrand
    const float *p0, *p1, *p2, *p3;
    bool odd = false;
    GaConst c0{};
    DeConst dc{};
    if constexpr (ALGO == A_GA_SBX_PM) {
        const U4 mb = rng.block((uint32_t)gen, P_GA_MATE, (uint32_t)(ie & ~1), 0u, 0u);
        const int ra = (int)g.modM.mod(pick(mb, (uint32_t)(il & 1)));
        const int rb = (int)g.modM.mod(pick(mb, (uint32_t)((il & 1) ^ 1)));
        p0 = L.X + (base + ra) * S::RS + off;
        p1 = L.X + (base + rb) * S::RS + off;
        p2 = p3 = p0;
        c0 = ga_const(a, td);
        odd = (il & 1) != 0;
    } else {
        const bool rand1 = (a.p.algo == A_DE_RAND_1_BIN);
        const DeMates mt = pair ? de_mates2(a, g, rng, gen, ie, h, first, next) : de_mates(a, g, rng, gen, ie);
        dc = de_const(a, td);
        dc.jr = mt.jrand - h;
        p0 = L.X + (base + (rand1 ? mt.r1 : il)) * S::RS + off;
        p1 = L.X + (base + mt.r2) * S::RS + off;
        p2 = L.X + (base + mt.r3) * S::RS + off;
        p3 = L.X + ie * S::RS + off;
    }
    // crossover draws, four blocks (32 genes) at a time
    constexpr int NCB = (KB + 1) / 2;
    U4 cbs[NCB < 4 ? NCB : 4], cbt[NCB > 4 ? NCB - 4 : 1];
    if constexpr (ALGO != A_GA_SBX_PM) rng.blocks(cbs, (uint32_t)gen, P_DE_CR, (uint32_t)ie, (uint32_t)h, 0u);
#pragma unroll
    for (int sb = 0; sb < KB; ++sb) {
        // past the dimension: finite slots, no steps (a uniform branch)
        if (kSkipBlock<KB> > 0 && sb >= kSkipBlock<KB> && 4 * sb >= g.Dh) {
#pragma unroll
            for (int e = 0; e < 4; ++e) tr[4 * sb + e] = 0.0f;
            continue;
        }
        float t[4];
        float4 vb, v2, v3, vi;
        if constexpr (ALGO == A_GA_SBX_PM) {
            ga_block(t, lds4(p0 + 4 * sb), lds4(p1 + 4 * sb), rng, gen, ie, sb, h, odd, g.D, c0);
        } else {
            if (sb == 8) rng.blocks(cbt, (uint32_t)gen, P_DE_CR, (uint32_t)ie, (uint32_t)h, 4u);
            vb = lds4(p0 + 4 * sb);
            v2 = lds4(p1 + 4 * sb);
            v3 = lds4(p2 + 4 * sb);
            vi = lds4(p3 + 4 * sb);
        }
        float4 q[NT];
#pragma unroll
        for (int jt = 0; jt < NT; ++jt) {
            if constexpr (kQGlobal<KB>) {
                q[jt] = qn[jt];
                if (sb + 1 < KB) qn[jt] = q_op(qrow, kQTiles, sb + 1, jt);
            } else {
                q[jt] = lds4(qrow + 32 * jt * S::RS + 4 * sb);
            }
        }
        const float4 o4 = lds4(orow + 4 * sb);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (ALGO != A_GA_SBX_PM)
                t[e] = de_gene(dc, f4(vb, e), f4(v2, e), f4(v3, e), f4(vi, e),
                               sb < 8 ? cbs[(sb >> 1) % (NCB < 4 ? NCB : 4)] : cbt[sb < 8 ? 0 : (sb >> 1) - 4], sb, e);
            tr[4 * sb + e] = t[e];
            // k-steps past the dimension add q * 0 of the zero padding: skipped
            if (sb < KB - 1 || 4 * sb + e < g.Dh) {
                const float w = t[e] - f4(o4, e);
#pragma unroll
                for (int jt = 0; jt < NT; ++jt)
                    acc[jt] = __builtin_amdgcn_mfma_f32_32x32x2f32(f4(q[jt], e), w, acc[jt], 0, 0, 0);
            }
        }
    }
    // the padded row groups are skipped for the two costliest epilogues only (measured:
    // the branch costs more than it saves for the others)
    // Q's rows past D are zero (in LDS zeroed at the epoch's start)
    return objective<NT, FUNC, FUNC == F_WEIERSTRASS || FUNC == F_SCHWEFEL || FUNC == F_REF_WEIERSTRASS, true>(
        acc, g.D, L.tab, h);
}

// Sixteen bytes at any float's address.
struct __attribute__((packed, aligned(4))) F4U {
    float x, y, z, w;
};

// Rows of an n x D row-major matrix in global memory to np rows of stride RS in the [even | odd]
// layout (gene d at (d & 1) HS + d / 2), nb blocks of eight genes each; zeros past the
// dimension and past row n.  A thread takes a block: two 16-byte loads and two 16-byte stores, B
// blocks in flight, so an epoch's start costs a latency or two and no division per gene.  A
// row's last block reads up to seven floats past the row: the arrays are allocated eight longer.
// What an epoch costs beside its generations (256 tasks, pop 128; with the ranking and the
// transfer): D = 50 29 to 24 us, D = 150 (wide kernel) 63 to 47.
template <int RS, int HS, int NTHR, int B>
__device__ __forceinline__ void stage_rows(float* dst, const float* __restrict__ src, int n, int np, int D, int nb,
                                           int tid) {
    const int di = NTHR / nb, dk = NTHR - di * nb;
    int i = tid / nb, k = tid - i * nb;
    while (i < np) {
        F4U v[B][2];
        int ii[B], kk[B];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            ii[b] = i;
            kk[b] = k;
            const F4U* s = reinterpret_cast<const F4U*>(src + (i < n && 8 * k < D ? (int64_t)i * D + 8 * k : 0));
            v[b][0] = s[0];
            v[b][1] = s[1];
            i += di;
            k += dk;
            if (k >= nb) {
                k -= nb;
                ++i;
            }
        }
#pragma unroll
        for (int b = 0; b < B; ++b) {
            if (ii[b] >= np) break;
            const int left = ii[b] < n ? D - 8 * kk[b] : 0;  // genes of the block
            const float4 ev = make_float4(left > 0 ? v[b][0].x : 0.0f, left > 2 ? v[b][0].z : 0.0f,
                                          left > 4 ? v[b][1].x : 0.0f, left > 6 ? v[b][1].z : 0.0f);
            const float4 od = make_float4(left > 1 ? v[b][0].y : 0.0f, left > 3 ? v[b][0].w : 0.0f,
                                          left > 5 ? v[b][1].y : 0.0f, left > 7 ? v[b][1].w : 0.0f);
            float* row = dst + (int64_t)ii[b] * RS + 4 * kk[b];
            *reinterpret_cast<float4*>(row) = ev;
            *reinterpret_cast<float4*>(row + HS) = od;
        }
    }
}

// The way back: n rows, row i at src + row(i), to an n x D row-major matrix.
template <int HS, int NTHR, int B, typename Row>
__device__ __forceinline__ void unstage_rows(float* __restrict__ dst, const float* src, Row row, int n, int D, int tid) {
    const int nb = (D + 7) >> 3, di = NTHR / nb, dk = NTHR - di * nb;
    int i = tid / nb, k = tid - i * nb;
    while (i < n) {
        float4 ev[B], od[B];
        int ii[B], kk[B];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            ii[b] = i;
            kk[b] = k;
            const float* r = src + (i < n ? row(i) + 4 * k : row(0));
            ev[b] = lds4(r);
            od[b] = lds4(r + HS);
            i += di;
            k += dk;
            if (k >= nb) {
                k -= nb;
                ++i;
            }
        }
#pragma unroll
        for (int b = 0; b < B; ++b) {
            if (ii[b] >= n) break;
            const int left = D - 8 * kk[b];
            float* o = dst + (int64_t)ii[b] * D + 8 * kk[b];
            const F4U lo{ev[b].x, od[b].x, ev[b].y, od[b].y}, hi{ev[b].z, od[b].z, ev[b].w, od[b].w};
            if (left >= 8) {
                reinterpret_cast<F4U*>(o)[0] = lo;
                reinterpret_cast<F4U*>(o)[1] = hi;
            } else {
                o[0] = lo.x;
                if (left > 1) o[1] = lo.y;
                if (left > 2) o[2] = lo.z;
                if (left > 3) o[3] = lo.w;
                if (left > 4) o[4] = hi.x;
                if (left > 5) o[5] = hi.y;
                if (left > 6) o[6] = hi.z;
            }
        }
    }
}

template <int KB>
__device__ __forceinline__ void load_half_row(float (&x)[4 * KB], const float* row) {
#pragma unroll
    for (int sb = 0; sb < KB; ++sb) {
        const float4 v = lds4(row + 4 * sb);
        x[4 * sb] = v.x; x[4 * sb + 1] = v.y; x[4 * sb + 2] = v.z; x[4 * sb + 3] = v.w;
    }
}

template <int KB>
__device__ __forceinline__ void store_half_row(float* row, const float (&x)[4 * KB]) {
#pragma unroll
    for (int sb = 0; sb < KB; ++sb)
        *reinterpret_cast<float4*>(row + 4 * sb) = make_float4(x[4 * sb], x[4 * sb + 1], x[4 * sb + 2], x[4 * sb + 3]);
}

// ---------------------------------------------------------------------------
// Population-level phases (all threads of the workgroup participate)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float key_of(float f) { return (f != f) ? __builtin_inff() : f; }

// ord[q m + rank] = i: the members of each island q ranked by (fitness, index).  Threads to
// spare share an individual's comparisons, two to eight adjacent lanes each.
template <int NTHR = kThreads>
__device__ __forceinline__ void rank_islands(const Lds& L, int pop, int m, int tid) {
    int sh = 0;
    while (sh < 3 && (pop << (sh + 1)) <= NTHR) ++sh;
    for (int t = tid; t < (pop << sh); t += NTHR) {
        const int i = t >> sh;
        const int q = i / m, base = q * m, il = i - base;
        const float fi = key_of(L.fit[i]);
        int r = 0;
#pragma unroll 8
        for (int p = t & ((1 << sh) - 1); p < m; p += 1 << sh) {
            const float fp = key_of(L.fit[base + p]);
            r += (fp < fi || (fp == fi && p < il)) ? 1 : 0;
        }
        for (int d = 1; d < (1 << sh); d <<= 1) r += __shfl_xor(r, d);
        if ((t & ((1 << sh) - 1)) == 0) L.ord[base + r] = i;
    }
}

template <int KB, int FUNC, int ALGO>
__device__ __forceinline__ void generation_step(const EpochArgs& a, const TaskDev& td, const Geo& g, const Lds& L,
                                                const Rng& rng, int gen, int tid, bool first, MateCache& next) {
    using S = Shape<KB>;
    const int wave = tid >> 6, lane = tid & 63, col = lane & 31, h = lane >> 5;
    const bool multi = g.ntiles > kThreads / 64;
    float tr[4 * KB];
    float fchild = 0.0f;
    int i_keep = -1;
    bool acc_keep = false;
    unsigned taken = 0u;  // multi: the wave's tiles whose trial the lane took
    for (int it = wave; it < g.ntiles; it += kThreads / 64) {
        const int i = it * 32 + col;
        const bool valid = i < g.pop;
        const int ie = valid ? i : 0;
        const float f = trial_eval<KB, FUNC, ALGO>(tr, a, td, g, L, rng, gen, ie, col, h, !multi, first, next);
        const bool accept = valid && (L.fit[i] >= f);
        if (multi) {
            if (accept) store_half_row<KB>(a.scratch + td.scr_off + (int64_t)i * S::RS + h * S::HS, tr);
            if (accept && h == 0) L.ftmp[i] = f;
            taken |= accept ? 1u << (it / (kThreads / 64)) : 0u;
        } else {
            i_keep = i;
            acc_keep = accept;
            fchild = f;
        }
    }
    __syncthreads();
    if (!multi) {
        if (i_keep >= 0 && acc_keep) {
            store_half_row<KB>(L.X + i_keep * S::RS + h * S::HS, tr);
            if (h == 0) L.fit[i_keep] = fchild;
        }
    } else {
        // each lane fetches the half rows that it left in scratch memory
        for (int it = wave; it < g.ntiles; it += kThreads / 64) {
            if (!((taken >> (it / (kThreads / 64))) & 1u)) continue;
            const int i = it * 32 + col;
            load_half_row<KB>(tr, a.scratch + td.scr_off + (int64_t)i * S::RS + h * S::HS);
            store_half_row<KB>(L.X + i * S::RS + h * S::HS, tr);
            if (h == 0) L.fit[i] = L.ftmp[i];
        }
    }
    __syncthreads();
}

// Cross-island resampling (reference SharedToGlobal + SelectFromBlocks).  The shuffles' draws
// and their remainders are formed by all threads, so the serial part of a shuffle is its swaps.
template <int KB, int NTHR = kThreads>
__device__ __forceinline__ void island_exchange(const EpochArgs& a, const Geo& g, const Lds& L, float* scr,
                                                const Rng& rng, int gen, int tid) {
    constexpr int RS = Shape<KB>::RS;
    const int n = a.p.n_islands, m = g.m, mb = (m + 3) >> 2;
    int* draw = reinterpret_cast<int*>(L.ftmp);
    for (int e = tid; e < n * mb; e += NTHR) {
        const int q = e / mb, b = e - q * mb;
        const U4 w = rng.block((uint32_t)gen, P_ISLX, (uint32_t)q, 0u, (uint32_t)b);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int k = m - 1 - (4 * b + c);
            if (k >= 0) draw[q * m + k] = (int)(pick(w, (uint32_t)c) % (uint32_t)(k + 1));
        }
    }
    for (int i = tid; i < g.pop; i += NTHR) L.aux[i] = i % m;
    __syncthreads();
    for (int q = tid; q < n; q += NTHR) {
        int* arr = L.aux + q * m;
        for (int k = m - 1; k >= 0; --k) {
            const int t = draw[q * m + k];
            const int tmp = arr[k];
            arr[k] = arr[t];
            arr[t] = tmp;
        }
    }
    __syncthreads();
    for (int i = tid; i < g.pop; i += NTHR) {  // inverse permutation
        const int q = i / m;
        L.ord[q * m + L.aux[i]] = i - q * m;
    }
    __syncthreads();
    // one island offset per slot k, shared by every island (the reference's
    // select_interval[iter * IPB + k] has no block term, SG-EMTF.cu:1227, :1597): each slot
    // is a rotation of the islands, so the exchange permutes the task's rows
    for (int i = tid; i < g.pop; i += NTHR) {
        const int q = i / m, k = i - q * m;
        const uint32_t w = rng.word((uint32_t)gen, P_ISLX, 0u, 1u, (uint32_t)k);
        const int src = (q + (int)(w % (uint32_t)n)) % n;
        L.aux[i] = src * m + L.ord[src * m + k];
    }
    __syncthreads();
    for (int i = tid; i < g.pop; i += NTHR) L.ftmp[i] = L.fit[L.aux[i]];
    if constexpr (NTHR == kThreads) {
        // rows in LDS: permuted through registers, as many columns at a time as eight 16-byte
        // blocks a thread hold of every row
        constexpr int B = 8;
        const int cols = B * NTHR / g.pop;
        for (int c0 = 0; c0 < RS / 4; c0 += cols) {
            const int nc = RS / 4 - c0 < cols ? RS / 4 - c0 : cols, total = g.pop * nc;
            float4 v[B];
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int e = tid + b * NTHR, row = e / nc, c = c0 + e - row * nc;
                if (e < total) v[b] = lds4(L.X + L.aux[row] * RS + 4 * c);
            }
            __syncthreads();
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int e = tid + b * NTHR, row = e / nc, c = c0 + e - row * nc;
                if (e < total) *reinterpret_cast<float4*>(L.X + row * RS + 4 * c) = v[b];
            }
        }
    } else {
        for (int e = tid; e < g.pop * (RS / 4); e += NTHR) {
            const int row = e / (RS / 4), c = 4 * (e - row * (RS / 4));
            *reinterpret_cast<float4*>(scr + 4 * e) = lds4(L.X + L.aux[row] * RS + c);
        }
        __syncthreads();
        for (int e = tid; e < g.pop * (RS / 4); e += NTHR)
            *reinterpret_cast<float4*>(L.X + 4 * e) = lds4(scr + 4 * e);
    }
    for (int i = tid; i < g.pop; i += NTHR) L.fit[i] = L.ftmp[i];
    __syncthreads();
}

// Intra-task island migration (reference IslandMigration).
template <int KB, int NTHR = kThreads>
__device__ __forceinline__ void island_migration(const EpochArgs& a, const Geo& g, const Lds& L, int tid) {
    constexpr int RS = Shape<KB>::RS;
    const int n = a.p.n_islands, m = g.m, kk = a.p.migrate_count;
    rank_islands<NTHR>(L, g.pop, m, tid);
    __syncthreads();
    for (int e = tid; e < n * kk; e += NTHR) {
        const int q = e / kk, j = e - q * kk, p = (q + 1) % n;
        const int src = L.ord[q * m + j], dst = L.ord[p * m + m - kk + j];
        L.aux[e] = (L.fit[src] < L.fit[dst]) ? 1 : 0;
    }
    __syncthreads();
    for (int e = tid; e < n * kk * RS; e += NTHR) {
        const int pr = e / RS, c = e - pr * RS;
        if (L.aux[pr]) {
            const int q = pr / kk, j = pr - q * kk, p = (q + 1) % n;
            const int src = L.ord[q * m + j], dst = L.ord[p * m + m - kk + j];
            L.X[dst * RS + c] = L.X[src * RS + c];
        }
    }
    for (int e = tid; e < n * kk; e += NTHR) {
        if (L.aux[e]) {
            const int q = e / kk, j = e - q * kk, p = (q + 1) % n;
            const int src = L.ord[q * m + j], dst = L.ord[p * m + m - kk + j];
            L.fit[dst] = L.fit[src];
        }
    }
    __syncthreads();
}

// Inter-task transfer at the start of an epoch (reference knowledgeTransfer).
template <int KB, int FUNC>
__device__ __forceinline__ void transfer_in(const EpochArgs& a, const TaskDev& td, const Geo& g, const Lds& L,
                                            const Rng& rng, int tid, int eg0) {
    using S = Shape<KB>;
    // draws at the task's own generation g0, the mailbox buffer by the handle's clock eg0
    const int k = a.p.transfer_count, TI = a.p.transfer_interval, g0 = eg0 - td.gen_base;
    const int wave = tid >> 6, lane = tid & 63, col = lane & 31, h = lane >> 5;
    rank_islands(L, g.pop, g.pop, tid);
    __syncthreads();
    const uint32_t wd = rng.word((uint32_t)g0, P_MIG, 0u, 0u, 0u);
    const int dn = pick_donor(a, (int)rng.task, wd);
    const TaskDev dd = a.tasks[dn];
    const float* mb = a.mailbox + (int64_t)((eg0 / TI) & 1) * a.mailbox_stride + dd.mb_off;
    const bool same_box = (dd.lo == td.lo && dd.hi == td.hi);
    const float rng_s = td.hi - td.lo, rng_d = dd.hi - dd.lo;
    const int ntc = (k + 31) / 32;
    for (int ct = wave; ct < ntc; ct += kThreads / 64) {
        const int j = ct * 32 + col;
        const bool valid = j < k;
        const int je = valid ? j : 0;
        // the donor's genes (of the build's every slot: the mailbox is allocated a longest row
        // longer), then the box and the draws where they matter, then one select a gene:
        // straight code, since every epoch fetches it anew
        const float* mrow = mb + (int64_t)je * dd.dim;
        const int dlim = (g.D < dd.dim ? g.D : dd.dim) - h;  // gene 2 q + h is transferable
        const float* own = L.X + L.ord[je] * S::RS + h * S::HS;
        float cand[S::HS];
        constexpr int VB = S::HS < 32 ? S::HS : 32;
#pragma unroll
        for (int q0 = 0; q0 < S::HS; q0 += VB) {
            float v[VB];
#pragma unroll
            for (int r = 0; r < VB; ++r) v[r] = mrow[2 * (q0 + r) + h];
            if (!same_box) {
#pragma unroll
                for (int r = 0; r < VB; ++r) {
                    const float t1 = v[r] - dd.lo;
                    const float t2 = t1 / rng_d;
                    const float t3 = t2 * rng_s;
                    v[r] = td.lo + t3;
                }
            }
            uint32_t take = 0xFFFFFFFFu;
            if (a.p.transfer_cr > 0.0f) {
                take = 0u;
#pragma unroll 1
                for (int b = 0; b < VB / 4; ++b) {
                    const U4 ub = rng.block((uint32_t)g0, P_XFER, (uint32_t)je, (uint32_t)h, (uint32_t)(q0 / 4 + b));
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        take |= uniform01(pick(ub, (uint32_t)e)) > a.p.transfer_cr ? 1u << (4 * b + e) : 0u;
                }
            }
#pragma unroll
            for (int r = 0; r < VB && q0 + r < S::HS; r += 4) {
                const float4 o4 = lds4(own + q0 + r);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    cand[q0 + r + e] = (2 * (q0 + r + e) < dlim && ((take >> (r + e)) & 1u)) ? v[r + e] : f4(o4, e);
            }
        }
        const float f = evaluate_tile<KB, FUNC>(cand, g, L, col, h);
        if (valid) {
            const int tgt = L.ord[g.pop - k + j];
            if (f < L.fit[tgt]) {
                store_half_row<KB>(L.X + tgt * S::RS + h * S::HS, cand);
                if (h == 0) L.fit[tgt] = f;
            }
        }
    }
    __syncthreads();
}

// d f / d z_j (0 for j >= D) of the point z in memory.
template <int FUNC>
__device__ __forceinline__ float dz_term(int j, const float* z, int D, const float* tab, const DzConst& kc, float pre,
                                         float suf) {
    if (j >= D) return 0.0f;
    const bool ros = FUNC == F_ROSENBROCK;
    return dz_elem<FUNC>(j, z[j], ros && j > 0 ? z[j - 1] : 0.0f, ros && j + 1 < D ? z[j + 1] : 0.0f, D, tab[j], kc, pre,
                         suf);
}

// z rows of tile jt for the lane's column from w = x - o (the lane's parity half, in
// registers): the k-steps of evaluate_tile's chain for that tile, whole blocks of four
// from the first, stopping after the block that holds step Dh - 1 (the steps past the
// dimension in it add zeros).
template <int KB>
__device__ __forceinline__ f16v tile_z(const float (&w)[4 * KB], const float* Q, int jt, int Dh, int col, int h) {
    using S = Shape<KB>;
    f16v acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const float* qrow = Q + (32 * jt + col) * S::RS + h * S::HS;
#pragma unroll
    for (int sb = 0; sb < KB; ++sb) {
        if (4 * sb >= Dh) break;
        const float4 q = lds4(qrow + 4 * sb);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(f4(q, e), w[4 * sb + e], acc, 0, 0, 0);
    }
    return acc;
}

// Polish staging per elite slot (floats): the point in the [even | odd] row layout, z,
// dz, the gradient and Griewank's prefix / suffix products (natural order), scalars,
// and the line search's candidates of one round (fitness, step) -- cpe each.
template <int KB>
struct PolishSlot {
    static constexpr int RS = Shape<KB>::RS, ZS = 32 * Shape<KB>::NT + 4;  // rows 16-byte aligned
    __host__ __device__ static constexpr int floats(int cpe) { return (RS + 5 * ZS + 16 + 2 * cpe + 3) & ~3; }
    static constexpr int kScratch = 128 + 128;  // after the slots: line-search sums, Rosenbrock rows
};

// Armijo polish of the top-k elites of one task, run between epochs after generation g1
// (restates the oracle's polish_task): from a Polyak step alpha = f / |g|^2 along -g,
// halve alpha until f(clamp(x - alpha g)) <= f - 1e-4 alpha |g|^2 (at most 24 halvings),
// take the step, repeat.  The elites go through in groups of 32 / cpe slots, all four
// waves working on every step of a group: each wave computes one 32-row tile of
// z = Q (x - o) (first step only) and of g = Q^T dz for every slot (column c holds slot
// c / cpe); dz is spread over all threads by (slot, dimension); the line search evaluates
// cpe halvings per slot per round (column c: halving round base + c mod cpe), each wave
// one row tile of the candidates' z, and the smallest accepted halving wins -- the step
// the one-at-a-time search takes; its z is kept as the next step's.  At a transfer
// boundary the task's elites are published afterwards.
template <int KB, int FUNC>
__device__ __forceinline__ void polish_body(const EpochArgs& a, float* smem, const TaskDev& td) {
    using S = Shape<KB>;
    constexpr int RS = S::RS, HS = S::HS, NT = S::NT, ZS = PolishSlot<KB>::ZS;
    constexpr int NW = kThreads / 64;
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, h = lane >> 5, wave = tid >> 6;
    Geo g{};
    g.D = td.dim;
    g.Dh = (g.D + 1) >> 1;
    g.pop = td.pop;
    g.popP = (g.pop + 31) & ~31;
    Lds L{};
    L.Q = smem;
    L.o = L.Q + 32 * NT * RS;
    L.tab = L.o + RS;
    L.fit = L.tab + 32 * NT;
    L.ord = reinterpret_cast<int*>(L.fit + g.popP);
    const int cpe = a.polish_cpe, nsl = 32 / cpe, PSZ = PolishSlot<KB>::floats(cpe);
    float* const slots = reinterpret_cast<float*>(L.ord + g.popP);
    float* const PS = slots + nsl * PSZ;  // the line search's running row sums, s1 | s2 per lane
    float* const PZ = PS + 128;           // Rosenbrock: row 0 of each tile per candidate
    static_assert(NT <= NW, "one row tile per wave in the line search");
    stage_rows<RS, HS, kThreads, 4>(L.Q, a.Q + td.q_off, g.D, 32 * NT, g.D, KB, tid);
    for (int d = tid; d < 32 * NT; d += kThreads) {
        if (d < 2 * HS) L.o[(d & 1) * HS + (d >> 1)] = d < g.D ? a.shift[td.v_off + d] : 0.0f;
        L.tab[d] = d < g.D ? a.tab[td.v_off + d] : 0.0f;
    }
    float* fitg = a.fit + td.fit_off;
    float* Xg = a.X + td.x_off;
    for (int i = tid; i < g.pop; i += kThreads) L.fit[i] = fitg[i];
    __syncthreads();
    rank_islands(L, g.pop, g.pop, tid);
    __syncthreads();
    const int K = a.p.polish_topk < g.pop ? a.p.polish_topk : g.pop;
    // per-slot views
    auto X = [&](int sl) { return slots + sl * PSZ; };
    auto Z = [&](int sl) { return X(sl) + RS; };
    auto DZ = [&](int sl) { return Z(sl) + ZS; };
    auto G = [&](int sl) { return DZ(sl) + ZS; };
    auto PRE = [&](int sl) { return G(sl) + ZS; };
    auto SUF = [&](int sl) { return PRE(sl) + ZS; };
    auto SF = [&](int sl) { return SUF(sl) + ZS; };  // f, g2, alpha0, ka, kb, fnew, alpha_ok
    auto SI = [&](int sl) { return reinterpret_cast<int*>(SF(sl) + 8); };  // active, done, first, elite
    auto CF = [&](int sl) { return SF(sl) + 16; };
    auto CA = [&](int sl) { return CF(sl) + cpe; };
    constexpr int kNone = 1 << 30;
    const int my_sl = col / cpe, sub = col - my_sl * cpe;
    for (int gb = 0; gb < K; gb += nsl) {
        const int ns = (K - gb) < nsl ? (K - gb) : nsl;
        for (int e = tid; e < nsl * 2 * HS; e += kThreads) {
            const int sl = e / (2 * HS), c = e - sl * (2 * HS);
            const int d = (c < HS) ? 2 * c : 2 * (c - HS) + 1;
            float v = 0.0f;
            if (sl < ns && d < g.D) v = Xg[(int64_t)L.ord[gb + sl] * g.D + d];
            X(sl)[c] = v;
        }
        for (int sl = tid; sl < nsl; sl += kThreads) {
            SF(sl)[0] = sl < ns ? L.fit[L.ord[gb + sl]] : 0.0f;
            SI(sl)[0] = sl < ns ? 1 : 0;
            SI(sl)[3] = sl < ns ? L.ord[gb + sl] : 0;
        }
        __syncthreads();
        for (int step = 0; step < a.p.polish_steps; ++step) {
            // z = Q (x - o) of every slot, one 32-row tile per wave (after the first step the
            // line search left it: an accepted slot's z, and an inactive slot's is unused)
            for (int jt = wave; step == 0 && jt < NT; jt += NW) {
                const float* xr = X(my_sl) + h * HS;
                float w[HS];
#pragma unroll
                for (int s4 = 0; s4 < HS; s4 += 4) {
                    const float4 x4 = lds4(xr + s4), o4 = lds4(L.o + h * HS + s4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) w[s4 + e] = f4(x4, e) - f4(o4, e);
                }
                const f16v acc = tile_z<KB>(w, L.Q, jt, g.Dh, col, h);
                if (sub == 0) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) Z(my_sl)[32 * jt + 8 * (r >> 2) + 4 * h + (r & 3)] = acc[r];
                }
            }
            __syncthreads();
            // per-slot factors: Ackley's, Griewank's prefix (even threads) / suffix (odd)
            // products; their per-dimension terms first, over all (slot, dimension) pairs
            // (into the dz and prefix rows, free until the dz pass), then the sums and
            // products in dimension order, one thread per slot and direction
            if constexpr (FUNC == F_ACKLEY || FUNC == F_GRIEWANK) {
                for (int e = tid; e < ns * g.D; e += kThreads) {
                    const int sl = e / g.D, j = e - sl * g.D;
                    const float zj = Z(sl)[j];
                    if constexpr (FUNC == F_ACKLEY) {
                        DZ(sl)[j] = zj * zj;
                        PRE(sl)[j] = sinpi_sq(zj);
                    } else {
                        DZ(sl)[j] = griewank_cos(zj, L.tab[j]);
                    }
                }
                __syncthreads();
            }
            if constexpr (FUNC == F_ACKLEY) {
                for (int sl = tid; sl < ns; sl += kThreads) {
                    float s1 = 0.0f, s2 = 0.0f;
                    for (int j = 0; j < g.D; ++j) {
                        s1 = s1 + DZ(sl)[j];
                        s2 = s2 + PRE(sl)[j];
                    }
                    const DzConst kc = ackley_const(s1, s2, g.D);
                    SF(sl)[3] = kc.ka;
                    SF(sl)[4] = kc.kb;
                }
                __syncthreads();
            }
            if constexpr (FUNC == F_GRIEWANK) {
                for (int e = tid; e < 2 * ns; e += kThreads) {
                    const int sl = e >> 1;
                    const float* c = DZ(sl);
                    float p = 1.0f;
                    if ((e & 1) == 0) {
                        for (int j = 0; j < g.D; ++j) {
                            PRE(sl)[j] = p;
                            p = p * c[j];
                        }
                    } else {
                        for (int j = g.D - 1; j >= 0; --j) {
                            SUF(sl)[j] = p;
                            p = p * c[j];
                        }
                    }
                }
                __syncthreads();
            }
            // dz of every (slot, dimension); zero past the dimension and for empty slots
            for (int e = tid; e < nsl * 2 * HS; e += kThreads) {
                const int sl = e / (2 * HS), j = e - sl * (2 * HS);
                float v = 0.0f;
                if (sl < ns) {
                    const DzConst kc{SF(sl)[3], SF(sl)[4]};
                    const bool gw = FUNC == F_GRIEWANK && j < g.D;
                    v = dz_term<FUNC>(j, Z(sl), g.D, L.tab, kc, gw ? PRE(sl)[j] : 0.0f, gw ? SUF(sl)[j] : 0.0f);
                }
                DZ(sl)[j] = v;
            }
            __syncthreads();
            // g = Q^T dz of every slot, one 32-row tile of dimensions per wave
            for (int dt = wave; dt < NT; dt += NW) {
                const float* dzr = DZ(my_sl);
                const int d = 32 * dt + col;
                f16v gacc;
#pragma unroll
                for (int r = 0; r < 16; ++r) gacc[r] = 0.0f;
                // blocks of four k-steps (rows j = 2 s2 + h); the steps past the dimension
                // in the last block add zeros (Q's padding rows and dz past D are zero)
                const float* qc = L.Q + (d & 1) * HS + (d >> 1);
#pragma unroll
                for (int sb = 0; sb < KB; ++sb) {
                    if (4 * sb >= g.Dh) break;
                    float qv[4], zv[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int j = 2 * (4 * sb + e) + h;
                        qv[e] = qc[j * RS];
                        zv[e] = dzr[j];
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) gacc = __builtin_amdgcn_mfma_f32_32x32x2f32(qv[e], zv[e], gacc, 0, 0, 0);
                }
                if (sub == 0) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) G(my_sl)[32 * dt + 8 * (r >> 2) + 4 * h + (r & 3)] = gacc[r];
                }
            }
            __syncthreads();
            // |g|^2 summed in dimension order, the Polyak step
            for (int sl = tid; sl < ns; sl += kThreads) {
                const float* gr = G(sl);
                float g2 = 0.0f;
                int d = 0;
                for (; d + 8 <= g.D; d += 8) {  // eight loads in flight, the chain in order
                    float v[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) v[k] = gr[d + k];
#pragma unroll
                    for (int k = 0; k < 8; ++k) g2 = fmaf(v[k], v[k], g2);
                }
                for (; d < g.D; ++d) g2 = fmaf(gr[d], gr[d], g2);
                const float f = SF(sl)[0];
                SF(sl)[1] = g2;
                SF(sl)[2] = f / g2;
                if (!(g2 > 0.0f) || !(f > 0.0f)) SI(sl)[0] = 0;
                SI(sl)[1] = 0;
                SI(sl)[2] = kNone;
            }
            __syncthreads();
            // Armijo rounds: halvings r0 .. r0 + cpe - 1 of every slot (column col: slot
            // col / cpe, halving r0 + col % cpe).  Wave w computes row tile w of the 32
            // candidates' z, and the objective's row sums run through the tiles in order:
            // wave w adds tile w's rows onto the sums wave w - 1 left in LDS, the last wave
            // finishes the fitness.  The accepted candidate's z is the next step's z.
            for (int r0 = 0;; r0 += cpe) {
                const int b = r0 + sub;
                const bool act = my_sl < ns && SI(my_sl)[0] && !SI(my_sl)[1];
                float alpha = SF(my_sl)[2];
                for (int q = 0; q < b; ++q) alpha = alpha * 0.5f;
                const float* xr = X(my_sl) + h * HS;
                const float* gr = G(my_sl);
                f16v acc;
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
                if (wave < NT) {
                    float w[HS];
#pragma unroll
                    for (int s4 = 0; s4 < HS; s4 += 4) {
                        const float4 x4 = lds4(xr + s4), o4 = lds4(L.o + h * HS + s4);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int s2 = s4 + e;
                            const float st = alpha * gr[2 * s2 + h];  // in the row (zeros past D)
                            const float xc = clampf(f4(x4, e) - st, td.lo, td.hi);
                            const float xn = (2 * s2 + h < g.D) ? xc : 0.0f;
                            w[s2] = xn - f4(o4, e);
                        }
                    }
                    acc = tile_z<KB>(w, L.Q, wave, g.Dh, col, h);
                    if (FUNC == F_ROSENBROCK && h == 0) PZ[32 * wave + col] = acc[0];
                }
                __syncthreads();
                float v1[16], v2[16];
                if (wave < NT) {
                    const float zn0 = (FUNC == F_ROSENBROCK && wave + 1 < NT) ? PZ[32 * (wave + 1) + col] : 0.0f;
                    tile_vals<FUNC>(acc, wave, g.D, L.tab, h, zn0, v1, v2);
                }
                float s1 = 0.0f, s2 = 0.0f;
                for (int st = 0; st < NT; ++st) {
                    if (wave == st) {
                        if (st > 0) {
                            s1 = PS[lane];
                            s2 = PS[64 + lane];
                        }
                        tile_sums<FUNC>(v1, v2, st, g.D, h, s1, s2);
                        if (st + 1 < NT) {
                            PS[lane] = s1;
                            PS[64 + lane] = s2;
                        }
                    }
                    if (st + 1 < NT) __syncthreads();
                }
                if (wave == NT - 1) {
                    const float fn = objective_tail<FUNC>(s1, s2, g.D, L.tab, h);
                    const float c1 = 1.0e-4f * alpha;
                    const float c2 = c1 * SF(my_sl)[1];
                    const float thr = SF(my_sl)[0] - c2;
                    if (act && b < 24 && fn <= thr && h == 0) {
                        CF(my_sl)[sub] = fn;
                        CA(my_sl)[sub] = alpha;
                        atomicMin(&SI(my_sl)[2], b);
                    }
                }
                __syncthreads();
                for (int sl = tid; sl < ns; sl += kThreads) {
                    const int fb = SI(sl)[2];
                    if (SI(sl)[0] && !SI(sl)[1] && fb != kNone) {
                        SI(sl)[1] = 1;
                        SF(sl)[5] = CF(sl)[fb - r0];
                        SF(sl)[6] = CA(sl)[fb - r0];
                    }
                }
                __syncthreads();
                // the accepted halving's lanes keep z = Q (x_new - o) for the next step (the
                // same MFMA chain the forward pass would run on the stepped point)
                if (wave < NT && my_sl < ns && SI(my_sl)[2] == b) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) Z(my_sl)[32 * wave + 8 * (r >> 2) + 4 * h + (r & 3)] = acc[r];
                }
                bool more = false;
                for (int sl = 0; sl < ns; ++sl) more = more || (SI(sl)[0] && !SI(sl)[1]);
                if (!more || r0 + cpe >= 24) break;
            }
            // accepted slots step to clamp(x - alpha g), the others stop
            for (int e = tid; e < ns * 2 * HS; e += kThreads) {
                const int sl = e / (2 * HS), c = e - sl * (2 * HS);
                if (SI(sl)[0] && SI(sl)[1]) {
                    const int d = (c < HS) ? 2 * c : 2 * (c - HS) + 1;
                    const float st = SF(sl)[6] * G(sl)[d];
                    X(sl)[c] = (d < g.D) ? clampf(X(sl)[c] - st, td.lo, td.hi) : 0.0f;
                }
            }
            __syncthreads();
            for (int sl = tid; sl < ns; sl += kThreads) {
                if (SI(sl)[0] && SI(sl)[1]) SF(sl)[0] = SF(sl)[5];
                else SI(sl)[0] = 0;
            }
            __syncthreads();
        }
        for (int e = tid; e < ns * g.D; e += kThreads) {
            const int sl = e / g.D, d = e - sl * g.D;
            Xg[(int64_t)SI(sl)[3] * g.D + d] = X(sl)[(d & 1) * HS + (d >> 1)];
        }
        for (int sl = tid; sl < ns; sl += kThreads) {
            L.fit[SI(sl)[3]] = SF(sl)[0];
            fitg[SI(sl)[3]] = SF(sl)[0];
        }
        __syncthreads();
    }
    if (a.publish) {
        rank_islands(L, g.pop, g.pop, tid);
        __syncthreads();
        const int k = a.p.transfer_count, TI = a.p.transfer_interval;
        float* mb = a.mailbox + (int64_t)((a.g1 / TI) & 1) * a.mailbox_stride + td.mb_off;
        for (int e = tid; e < k * g.D; e += kThreads) {
            const int r = e / g.D, d = e - r * g.D;
            mb[e] = Xg[(int64_t)L.ord[r] * g.D + d];
        }
    }
}

template <int KB>
__global__ __launch_bounds__(kThreads) void polish_kernel(EpochArgs a, const int* __restrict__ order) {
    extern __shared__ float smem[];
    const TaskDev td = a.tasks[order[blockIdx.x]];
    switch (td.func) {
    case F_SPHERE: polish_body<KB, F_SPHERE>(a, smem, td); break;
    case F_ROSENBROCK: polish_body<KB, F_ROSENBROCK>(a, smem, td); break;
    case F_ACKLEY: polish_body<KB, F_ACKLEY>(a, smem, td); break;
    case F_RASTRIGIN: polish_body<KB, F_RASTRIGIN>(a, smem, td); break;
    case F_GRIEWANK: polish_body<KB, F_GRIEWANK>(a, smem, td); break;
    case F_WEIERSTRASS: polish_body<KB, F_WEIERSTRASS>(a, smem, td); break;
    case F_SCHWEFEL: polish_body<KB, F_SCHWEFEL>(a, smem, td); break;
    case F_ELLIPTIC: polish_body<KB, F_ELLIPTIC>(a, smem, td); break;
    default: break;
    }
}

// Thread 0's bounded wait for *p >= v under the persistent schedule (device-scope acquire
// loads; false once the handle's error flag is set or the wait runs out, which sets it).
__device__ __noinline__ bool persist_wait(const int32_t* p, int32_t v, const PersistArgs& pa) {
    const uint64_t t0 = wall_clock64();
    for (;;) {
        if (__hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) >= v) return true;
        if (__hip_atomic_load(pa.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
        if ((int64_t)(wall_clock64() - t0) > pa.wait_ticks) {
            __hip_atomic_store(pa.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        __builtin_amdgcn_s_sleep(8);
    }
}

// PERSIST: the epoch is item (pe, task) of a persistent launch -- it counts itself in
// pa->reads[pe] once past its mailbox read, and waits for every item of epoch pe - 1 to
// be past theirs before it overwrites their mailbox buffer.
template <int KB, int FUNC, int ALGO, bool PERSIST = false>
__device__ __forceinline__ void epoch_body(const EpochArgs& a, float* smem, const int task, const TaskDev& td,
                                           const PersistArgs* pa = nullptr, int pe = 0, int pg0 = 0, int pg1 = 0,
                                           int ppub = 0) {
    // the epoch's generations and publish flag: the launch's, or the persistent item's
    const int eg0 = PERSIST ? pg0 : a.g0, eg1 = PERSIST ? pg1 : a.g1, epub = PERSIST ? ppub : a.publish;
    using S = Shape<KB>;
    constexpr int RS = S::RS, HS = S::HS, NT = S::NT;
    const int tid = threadIdx.x;
    Geo g;
    g.D = td.dim;
    g.Dh = (g.D + 1) >> 1;
    g.pop = td.pop;
    g.popP = (g.pop + 31) & ~31;
    g.ntiles = g.popP / 32;
    g.m = g.pop / (a.p.n_islands > 0 ? a.p.n_islands : 1);
    g.modD.init((uint32_t)g.D);
    g.modM.init((uint32_t)g.m);
    Lds L;
    L.X = smem;
    L.Q = kQGlobal<KB> ? const_cast<float*>(a.Qw + td.qw_off) : L.X + g.popP * RS;
    L.o = kQGlobal<KB> ? L.X + g.popP * RS : L.Q + 32 * NT * RS;
    L.tab = L.o + RS;
    L.fit = L.tab + 32 * NT;
    L.ftmp = L.fit + g.popP;
    L.ord = reinterpret_cast<int*>(L.ftmp + g.popP);
    L.aux = L.ord + g.popP;
    const Rng rng{a.p.seed_lo, a.p.seed_hi, (uint32_t)task};
    const int lane = tid & 63, col = lane & 31, h = lane >> 5, wave = tid >> 6;

    if (a.init) {
        for (int e = tid; e < g.popP * RS; e += kThreads) L.X[e] = 0.0f;
        __syncthreads();
    } else {
        stage_rows<RS, HS, kThreads, 4>(L.X, a.X + td.x_off, g.pop, g.pop, g.D, KB, tid);
    }
    if constexpr (!kQGlobal<KB>) stage_rows<RS, HS, kThreads, 4>(L.Q, a.Q + td.q_off, g.D, 32 * NT, g.D, KB, tid);
    for (int d = tid; d < 32 * NT; d += kThreads) {
        if (d < 2 * HS) L.o[(d & 1) * HS + (d >> 1)] = d < g.D ? a.shift[td.v_off + d] : 0.0f;
        L.tab[d] = d < g.D ? a.tab[td.v_off + d] : 0.0f;
    }
    if (a.init) {
        const float lo = td.lo, rng_ = td.hi - td.lo;
        for (int e = tid; e < g.pop * g.D; e += kThreads) {
            const int i = e / g.D, d = e - i * g.D;
            const float u = uniform01(rng.word(0u, P_INIT, (uint32_t)i, 0u, (uint32_t)d));
            const float t1 = u * rng_;
            L.X[i * RS + (d & 1) * HS + (d >> 1)] = t1 + lo;
        }
        __syncthreads();
        for (int it = wave; it < g.ntiles; it += kThreads / 64) {
            const int i = it * 32 + col;
            float x[HS];
            load_half_row<KB>(x, L.X + i * RS + h * HS);
            const float f = evaluate_tile<KB, FUNC>(x, g, L, col, h);
            if (i < g.pop && h == 0) L.fit[i] = f;
        }
    } else {
        for (int i = tid; i < g.pop; i += kThreads) L.fit[i] = a.fit[td.fit_off + i];
    }
    __syncthreads();

    const int TI = a.p.transfer_interval;
    if (transfer_now(a, td, eg0)) transfer_in<KB, FUNC>(a, td, g, L, rng, tid, eg0);
    if constexpr (PERSIST) {
        __syncthreads();
        if (tid == 0) __hip_atomic_fetch_add(pa->reads + pe, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }

    const bool islands = a.p.n_islands > 1;
    bool first = true;  // of two generations whose mates are drawn together (one tile per wave)
    MateCache next{0u, 0u};
    for (int gen = eg0 - td.gen_base + 1; gen <= eg1 - td.gen_base; ++gen, first = !first) {
        if (islands && a.p.exchange_interval > 0 && gen % a.p.exchange_interval == 0)
            island_exchange<KB>(a, g, L, a.scratch + td.scr_off, rng, gen, tid);
        generation_step<KB, FUNC, ALGO>(a, td, g, L, rng, gen, tid, first, next);
        if (islands && a.p.migrate_interval > 0 && a.p.migrate_count > 0 && gen % a.p.migrate_interval == 0)
            island_migration<KB>(a, g, L, tid);
    }

    // ranked before anything is stored: a barrier waits for the stores
    if (epub) {
        rank_islands(L, g.pop, g.pop, tid);
        __syncthreads();
    }
    unstage_rows<HS, kThreads, 4>(a.X + td.x_off, L.X, [](int i) { return i * RS; }, g.pop, g.D, tid);
    for (int i = tid; i < g.pop; i += kThreads) a.fit[td.fit_off + i] = L.fit[i];
    if (epub) {
        if constexpr (PERSIST) {
            __shared__ int s_pub;
            if (tid == 0) s_pub = (pe == 0 || persist_wait(pa->reads + pe - 1, a.n_tasks, *pa)) ? 1 : 0;
            __syncthreads();
            if (!s_pub) return;  // the error flag is set: the launch drains
        }
        const int k = a.p.transfer_count;
        float* mb = a.mailbox + (int64_t)((eg1 / TI) & 1) * a.mailbox_stride + td.mb_off;
        for (int e = tid; e < k * g.D; e += kThreads) {
            const int r = e / g.D, d = e - r * g.D;
            mb[e] = L.X[L.ord[r] * RS + (d & 1) * HS + (d >> 1)];
        }
    }
}

// One workgroup per task; `order` lists the tasks longest-first so the
// expensive objectives are dispatched before the cheap ones fill the gaps.
// Register budget: with KB <= 8 (dims <= 64) three 4-wave workgroups fit in LDS per
// CU, so the allocator is asked for 3 waves per SIMD (<= 168 VGPR+AGPR); of the larger
// rows two fit (256).
#if !defined(EMTF_WAVES_PER_EU) && defined(EMTF_KB)
#if EMTF_KB <= 8
#define EMTF_WAVES_PER_EU 3
#else
#define EMTF_WAVES_PER_EU 2
#endif
#endif
#ifdef EMTF_WAVES_PER_EU
#define EMTF_OCCUPANCY __attribute__((amdgpu_waves_per_eu(EMTF_WAVES_PER_EU, EMTF_WAVES_PER_EU)))
#else
#define EMTF_OCCUPANCY
#endif

template <int KB, int ALGO>
__global__ __launch_bounds__(kThreads) EMTF_OCCUPANCY void island_epoch_kernel(EpochArgs a, const int* __restrict__ order) {
    extern __shared__ float smem[];
    rebase_epoch(a);
    const int task = order[blockIdx.x];
    const TaskDev td = a.tasks[task];
    if (!runs_epoch(a, td)) return;
    switch (td.func) {
    case F_SPHERE: epoch_body<KB, F_SPHERE, ALGO>(a, smem, task, td); break;
    case F_ROSENBROCK: epoch_body<KB, F_ROSENBROCK, ALGO>(a, smem, task, td); break;
    case F_ACKLEY: epoch_body<KB, F_ACKLEY, ALGO>(a, smem, task, td); break;
    case F_RASTRIGIN: epoch_body<KB, F_RASTRIGIN, ALGO>(a, smem, task, td); break;
    case F_GRIEWANK: epoch_body<KB, F_GRIEWANK, ALGO>(a, smem, task, td); break;
    case F_WEIERSTRASS: epoch_body<KB, F_WEIERSTRASS, ALGO>(a, smem, task, td); break;
    case F_SCHWEFEL: epoch_body<KB, F_SCHWEFEL, ALGO>(a, smem, task, td); break;
    case F_ELLIPTIC: epoch_body<KB, F_ELLIPTIC, ALGO>(a, smem, task, td); break;
    case F_REF_ACKLEY: epoch_body<KB, F_REF_ACKLEY, ALGO>(a, smem, task, td); break;
    case F_REF_RASTRIGIN: epoch_body<KB, F_REF_RASTRIGIN, ALGO>(a, smem, task, td); break;
    case F_REF_GRIEWANK: case F_REF_GRIEWANK_GA: epoch_body<KB, F_REF_GRIEWANK, ALGO>(a, smem, task, td); break;
    case F_REF_WEIERSTRASS: epoch_body<KB, F_REF_WEIERSTRASS, ALGO>(a, smem, task, td); break;
    case F_REF_SCHWEFEL: epoch_body<KB, F_SCHWEFEL, ALGO>(a, smem, task, td); break;
    default: break;
    }
}


// The persistent schedule: generations pa.G0+1 .. pa.G1 of every task in one launch of
// n_epochs x n_tasks workgroups.  Each workgroup takes the next item (epoch e, task
// order[i]), e-major, from pa.next in the order the workgroups start (not by blockIdx), so
// every item it may wait on was taken earlier by a workgroup that is running; it waits for
// its task's epoch e - 1 and, at a transfer boundary, for its donor's (the one transfer_in
// draws), runs the epoch (PERSIST hooks: the mailbox read count and the wait before
// publishing) and releases pa.stamp[task] = e + 1.  No wait targets a later item, so the
// launch finishes whatever the number of resident workgroups; every wait is bounded.
template <int KB, int ALGO>
__global__ __launch_bounds__(kThreads) EMTF_OCCUPANCY void island_persistent_kernel(EpochArgs a, PersistArgs pa,
                                                                                   const int* __restrict__ order) {
    extern __shared__ float smem[];
    __shared__ int s_item, s_ok;
    const int tid = threadIdx.x;
    const int TI = a.p.transfer_interval;
    const bool xfer = TI > 0 && a.n_tasks > 1 && a.p.transfer_count > 0;
    const int n_items = pa.n_epochs * a.n_tasks;
    {
        if (tid == 0) s_item = __hip_atomic_fetch_add(pa.next, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const int item = s_item;
        if (item >= n_items) return;
        const int e = item / a.n_tasks;
        const int task = order[item - e * a.n_tasks];
        int g0, g1, pub;
        if (xfer) {
            const int b0 = pa.G0 / TI;  // epochs end at the transfer boundaries
            g0 = e == 0 ? pa.G0 : (b0 + e) * TI;
            g1 = min((b0 + e + 1) * TI, pa.G1);
            pub = g1 % TI == 0 ? 1 : 0;
        } else {
            g0 = pa.G0;
            g1 = pa.G1;
            pub = 0;
        }
        const TaskDev td = a.tasks[task];
        if (tid == 0) {
            bool ok = persist_wait(pa.stamp + task, e, pa);
            if (ok && transfer_now(a, td, g0)) {
                const Rng rng{a.p.seed_lo, a.p.seed_hi, (uint32_t)task};
                const uint32_t wd = rng.word((uint32_t)(g0 - td.gen_base), P_MIG, 0u, 0u, 0u);
                ok = persist_wait(pa.stamp + pick_donor(a, task, wd), e, pa);
            }
            s_ok = ok ? 1 : 0;
        }
        __syncthreads();
        if (!s_ok) return;  // the error flag is set: the launch drains
        // (the waits' acquire loads and the stamp's release store, with the fence and the
        // workgroup barriers around them, order the rows, fitness and mailbox across workgroups)
        switch (td.func) {
        case F_SPHERE: epoch_body<KB, F_SPHERE, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_ROSENBROCK: epoch_body<KB, F_ROSENBROCK, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_ACKLEY: epoch_body<KB, F_ACKLEY, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_RASTRIGIN: epoch_body<KB, F_RASTRIGIN, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_GRIEWANK: epoch_body<KB, F_GRIEWANK, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_WEIERSTRASS: epoch_body<KB, F_WEIERSTRASS, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_SCHWEFEL: epoch_body<KB, F_SCHWEFEL, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_ELLIPTIC: epoch_body<KB, F_ELLIPTIC, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_REF_ACKLEY: epoch_body<KB, F_REF_ACKLEY, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_REF_RASTRIGIN: epoch_body<KB, F_REF_RASTRIGIN, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_REF_GRIEWANK: case F_REF_GRIEWANK_GA:
            epoch_body<KB, F_REF_GRIEWANK, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub);
            break;
        case F_REF_WEIERSTRASS: epoch_body<KB, F_REF_WEIERSTRASS, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        case F_REF_SCHWEFEL: epoch_body<KB, F_SCHWEFEL, ALGO, true>(a, smem, task, td, &pa, e, g0, g1, pub); break;
        default: break;
        }
        // every wave's rows, fitness and elites are in memory before the stamp: the barrier
        // alone does not wait for the other waves' stores
        __threadfence();
        __syncthreads();
        if (tid == 0 && __hip_atomic_load(pa.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
            __hip_atomic_store(pa.stamp + task, e + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
}

#if defined(EMTF_WIDE_NT)
// ---------------------------------------------------------------------------
// Wide tasks: dimensions up to 32 NT, any population.  The population's rows live in global
// memory (a task's working set stays L2-resident while its workgroup runs), two rows per
// individual: the individual and its trial, which change roles when the trial is accepted
// (L.off[i], the individual's row).  LDS keeps the task's Q image where it fits (QL; else it
// is read from L2), o, the per-dimension table and the per-individual arrays.  A generation
// of the eight waves has three phases:
//   mates   one thread per individual draws its mates and leaves their row offsets in LDS;
//   trials  one thread per (individual, parity half, octet of genes): a Philox block's eight
//           crossover draws, 32 contiguous bytes of each parent row -- with the matrix
//           instructions' mapping (an individual per column) a load touched 64 rows for 16
//           bytes of each, and the rows went through L1 eight times over;
//   fitness z = Q w by v_mfma_f32_32x32x2_f32 over the trial rows, then the objective.  A wave
//           per tile of 32 individuals where there are five tiles or more, else the tile's row
//           tiles are dealt to 2, 4 or 8 waves: each computes the terms of its rows, and the
//           sums run through the waves in row order (so the bits are those of one wave).
// What bounds it: for large populations the fitness phase's MFMA (32 NT cycles a gene and tile)
// and then the trials' row traffic (256 tasks of D = 150, pop 256 read and write 240 MB a
// generation, 5 TB/s through L2 and the last-level cache), for small ones barriers and latencies.
// An epoch of 20 generations of 256 sphere tasks, against a kernel that formed the trials in the
// matrix instructions' mapping (its fastest build): D = 150, pop 32 / 128 / 256 0.495 / 0.661 /
// 1.365 to 0.257 / 0.609 / 1.017 ms; D = 180, pop 128 / 256 0.828 / 1.701 to 0.717 / 1.321; D = 200
// (Q from L2) 1.819 / 4.087 to 1.004 / 1.700.  Rows use the LDS path's [even | odd]
// layout with HS = 16 NT; the gene order of every fma chain is the LDS path's, with the padded
// k-steps past the dimension skipped (they would add +0).
// ---------------------------------------------------------------------------
constexpr int kWideThreads = 512, kWideWaves = kWideThreads / 64;

template <int NT>
using WShape = Shape<4 * NT>;

// acc[jt] += Q rows (32 jt + col) x (4 genes of one block of the lane's half)
template <int NT>
__device__ __forceinline__ void mfma_q(f16v (&acc)[NT], const float4 (&q)[NT], const float4& w4) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
            acc[jt] = __builtin_amdgcn_mfma_f32_32x32x2f32(f4(q[jt], e), f4(w4, e), acc[jt], 0, 0, 0);
}

template <int NT>
__device__ __forceinline__ void mfma_block(f16v (&acc)[NT], const float* ql, const float4& w4, int sb) {
    float4 q[NT];
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) q[jt] = q_op(ql, NT, sb, jt);
    mfma_q<NT>(acc, q, w4);
}

__device__ __forceinline__ float4 sub4(const float4& x, const float4& o) {
    return make_float4(x.x - o.x, x.y - o.y, x.z - o.z, x.w - o.w);
}

template <int NT>
__device__ __forceinline__ void zero_acc(f16v (&acc)[NT]) {
#pragma unroll
    for (int jt = 0; jt < NT; ++jt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[jt][r] = 0.0f;
}

// f of the lane's row (its parity half at row_h) read from memory
template <int NT, int FUNC>
__device__ __forceinline__ float wide_eval_row(const float* row_h, const Geo& g, const Lds& L, int col, int h, int nsb) {
    using S = WShape<NT>;
    f16v acc[NT];
    zero_acc<NT>(acc);
    const float* ql = L.Q + 4 * (32 * h + col);
    const float* orow = L.o + h * S::HS;
    for (int sb = 0; sb < nsb; ++sb) mfma_block<NT>(acc, ql, sub4(lds4(row_h + 4 * sb), lds4(orow + 4 * sb)), sb);
    return objective<NT, FUNC, true>(acc, g.D, L.tab, h);
}

// LDS of a wide task behind the Q image (QL).  `shared` holds the mates while trials are formed,
// the split sums while fitness is computed, and the scratch, rank and flag arrays between.
struct WideLds {
    int* off;    // popP: the individual's row, in floats from the first row
    int4* mate;  // popP: row offsets of the three mates (GA: two) and of the individual
    int* jr;     // popP: jrand
    float* ps;   // 4 tiles x 128: running sums s1 | s2 per lane
    float* pz;   // 8 waves x 32: Rosenbrock, row 0 of the wave's first row tile
};

__host__ __device__ inline int wide_lds_floats(int nt, int pop, bool ql) {
    const int RS = 32 * nt + 4, popP = (pop + 31) & ~31, sh = 5 * popP > 1280 ? 5 * popP : 1280;
    return (ql ? 1024 * nt * nt : 0) + RS + 32 * nt + 2 * popP + sh;
}

// Mates of every individual as row offsets.
template <int ALGO>
__device__ __forceinline__ void wide_mates(const EpochArgs& a, const Geo& g, const WideLds& W, const Rng& rng, int gen,
                                           int tid) {
    for (int i = tid; i < g.pop; i += kWideThreads) {
        const int il = (int)g.modM.mod((uint32_t)i), base = i - il;
        int4 m;
        if constexpr (ALGO == A_GA_SBX_PM) {
            const U4 mb = rng.block((uint32_t)gen, P_GA_MATE, (uint32_t)(i & ~1), 0u, 0u);
            m.x = W.off[base + (int)g.modM.mod(pick(mb, (uint32_t)(il & 1)))];
            m.y = W.off[base + (int)g.modM.mod(pick(mb, (uint32_t)((il & 1) ^ 1)))];
            m.z = 0;
        } else {
            const DeMates mt = de_mates(a, g, rng, gen, i);
            m.x = W.off[a.p.algo == A_DE_RAND_1_BIN ? base + mt.r1 : i];
            m.y = W.off[base + mt.r2];
            m.z = W.off[base + mt.r3];
            W.jr[i] = mt.jrand;
        }
        m.w = W.off[i];
        W.mate[i] = m;
    }
}

// Trial rows: unit e = (individual i, half h, octet o), U units per individual; i0, r0: the
// thread's first unit, di, dr: its step.
template <int NT, int ALGO>
__device__ __forceinline__ void wide_trials(const EpochArgs& a, const TaskDev& td, const Geo& g, float* X,
                                            const WideLds& W, const Rng& rng, int gen, int i0, int r0, int U) {
    using S = WShape<NT>;
    constexpr int RS = S::RS, HS = S::HS;
    const int noct = U >> 1, di = kWideThreads / U, dr = kWideThreads - di * U;
    int i = i0, r = r0;
    DeConst dc{};
    GaConst gc{};
    if constexpr (ALGO == A_GA_SBX_PM) gc = ga_const(a, td);
    else dc = de_const(a, td);
    while (i < g.pop) {
        const int h = r >= noct ? 1 : 0, o = r - (h ? noct : 0), c = h * HS + 8 * o;
        const int4 m = W.mate[i];
        float* dst = X + (2 * i + g.popP) * RS - m.w + c;  // the individual's other row
        const float *pa = X + m.x + c, *pb = X + m.y + c;
        float4 out[2];
        if constexpr (ALGO == A_GA_SBX_PM) {
#pragma unroll 1
            for (int b = 0; b < 2; ++b) {
                float t[4];
                ga_block(t, lds4(pa + 4 * b), lds4(pb + 4 * b), rng, gen, i, 2 * o + b, h, (i & 1) != 0, g.D, gc);
                *reinterpret_cast<float4*>(dst + 4 * b) = make_float4(t[0], t[1], t[2], t[3]);
            }
        } else {
            const float *pc = X + m.z + c, *pi = X + m.w + c;
            float4 va[2], vb[2], vc[2], vi[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                va[b] = lds4(pa + 4 * b);
                vb[b] = lds4(pb + 4 * b);
                vc[b] = lds4(pc + 4 * b);
                vi[b] = lds4(pi + 4 * b);
            }
            const U4 cb = rng.block((uint32_t)gen, P_DE_CR, (uint32_t)i, (uint32_t)h, (uint32_t)o);
            dc.jr = W.jr[i] - h - 16 * o;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                float t[4];
                de_block(t, va[b], vb[b], vc[b], vi[b], cb, b, dc);
                out[b] = make_float4(t[0], t[1], t[2], t[3]);
            }
#pragma unroll
            for (int b = 0; b < 2; ++b) *reinterpret_cast<float4*>(dst + 4 * b) = out[b];
        }
        i += di;
        r += dr;
        if (r >= U) {
            r -= U;
            ++i;
        }
    }
}

// z rows of R row tiles from jt0 of the lane's trial row (its parity half at trow, global
// memory): four gene blocks (64 bytes) of the row loaded at a time, the next four while these
// are multiplied.  Row tiles past the last repeat it (their z is not used).
template <int NT, int R, bool QL>
__device__ __forceinline__ void wide_z(f16v (&acc)[R], const float* trow, const float* Q, int jt0, const float* orow,
                                       int col, int h, int nsb) {
    zero_acc<R>(acc);
    const float* qt[R];
#pragma unroll
    for (int r = 0; r < R; ++r) qt[r] = Q + 4 * (32 * h + col) + 256 * (jt0 + r < NT ? jt0 + r : NT - 1);
    float4 nb[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) nb[k] = lds4(trow + 4 * k);
    float4 q[R];
    if constexpr (!QL) {
#pragma unroll
        for (int r = 0; r < R; ++r) q[r] = q_op(qt[r], NT, 0, 0);
    }
#pragma unroll 1
    for (int s0 = 0; s0 < nsb; s0 += 4) {
        float4 b[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) b[k] = nb[k];
        if (s0 + 4 < nsb) {
#pragma unroll
            for (int k = 0; k < 4; ++k) nb[k] = lds4(trow + 4 * (s0 + 4 + k));
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int sb = s0 + k;
            if (k > 0 && sb >= nsb) break;
            const float4 w = sub4(b[k], lds4(orow + 4 * sb));
            if constexpr (QL) {
#pragma unroll
                for (int r = 0; r < R; ++r) q[r] = q_op(qt[r], NT, sb, 0);
                mfma_q<R>(acc, q, w);
            } else {
                // Q from L2: a row tile's four steps, then its operands of the next block
                // into the same registers
#pragma unroll
                for (int r = 0; r < R; ++r) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[r] = __builtin_amdgcn_mfma_f32_32x32x2f32(f4(q[r], e), f4(w, e), acc[r], 0, 0, 0);
                    if (sb + 1 < nsb) q[r] = q_op(qt[r], NT, sb + 1, 0);
                }
            }
        }
    }
}

// The individual's trial replaces it when its fitness is no worse.
__device__ __forceinline__ void wide_select(const Geo& g, const Lds& L, const WideLds& W, int RS, int i, int h, float f) {
    if (i < g.pop && h == 0 && L.fit[i] >= f) {
        L.fit[i] = f;
        W.off[i] = (2 * i + g.popP) * RS - W.off[i];
    }
}

// Fitness of the trials, a wave per tile.
template <int NT, int FUNC, bool QL>
__device__ __forceinline__ void wide_fitness(const Geo& g, const Lds& L, const WideLds& W, int wave, int col, int h, int nsb) {
    using S = WShape<NT>;
    for (int it = wave; it < g.ntiles; it += kWideWaves) {
        const int i = it * 32 + col;
        const float* trow = L.X + (2 * i + g.popP) * S::RS - W.off[i] + h * S::HS;
        f16v acc[NT];
        wide_z<NT, NT, QL>(acc, trow, L.Q, 0, L.o + h * S::HS, col, h, nsb);
        const float f = objective<NT, FUNC, true>(acc, g.D, L.tab, h);
        wide_select(g, L, W, S::RS, i, h, f);
    }
}

// Fitness of the trials of at most four tiles, each tile's row tiles dealt R at a time to
// kWideWaves / ... waves (SP waves per tile, wave = SP tile + group).  Every wave takes part in
// the barriers.
template <int NT, int FUNC, bool QL, int R, int SP>
__device__ __forceinline__ void wide_fitness_split(const Geo& g, const Lds& L, const WideLds& W, int wave, int lane, int col,
                                                   int h, int nsb) {
    using S = WShape<NT>;
    constexpr int NG = (NT + R - 1) / R;  // groups of row tiles
    static_assert(NG <= SP && R * SP >= NT, "every row tile has a wave");
    const int it = wave / SP, grp = wave % SP;
    const bool active = it < g.ntiles && grp < NG;
    const int i = (it < g.ntiles ? it : 0) * 32 + col, jt0 = grp * R;
    f16v acc[R];
    float v1[R][16], v2[R][16];
    if (active) {
        const float* trow = L.X + (2 * i + g.popP) * S::RS - W.off[i] + h * S::HS;
        wide_z<NT, R, QL>(acc, trow, L.Q, jt0, L.o + h * S::HS, col, h, nsb);
        if (FUNC == F_ROSENBROCK && h == 0) W.pz[32 * wave + col] = acc[0][0];
    }
    if constexpr (FUNC == F_ROSENBROCK) __syncthreads();
    if (active) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float zn0 = 0.0f;  // row 32 (jt + 1) of z
            if constexpr (FUNC == F_ROSENBROCK) {
                if (r + 1 < R) zn0 = __shfl_xor(acc[r + 1 < R ? r + 1 : r][0], 32);
                else if (grp + 1 < NG) zn0 = W.pz[32 * (wave + 1) + col];
            }
            if (jt0 + r < NT) tile_vals<FUNC>(acc[r], jt0 + r, g.D, L.tab, h, zn0, v1[r], v2[r]);
        }
    }
    for (int st = 0; st < NG; ++st) {
        if (active && grp == st) {
            float s1, s2;
            sums_start<FUNC>(s1, s2);
            if (st > 0) {
                s1 = W.ps[128 * it + lane];
                s2 = W.ps[128 * it + 64 + lane];
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (jt0 + r < NT) tile_sums<FUNC>(v1[r], v2[r], jt0 + r, g.D, h, s1, s2);
            if (st + 1 < NG) {
                W.ps[128 * it + lane] = s1;
                W.ps[128 * it + 64 + lane] = s2;
            } else {
                const float f = objective_tail<FUNC>(s1, s2, g.D, L.tab, h);
                wide_select(g, L, W, S::RS, i, h, f);
            }
        }
        if (st + 1 < NG) __syncthreads();
    }
}

// Every individual's row back in the first set of rows (before phases that move rows).
template <int NT>
__device__ __forceinline__ void wide_gather(const Geo& g, const Lds& L, const WideLds& W, int tid) {
    constexpr int RS = WShape<NT>::RS;
    for (int e = tid; e < g.pop * (RS / 4); e += kWideThreads) {
        const int i = e / (RS / 4), c = 4 * (e - i * (RS / 4));
        if (W.off[i] != i * RS) *reinterpret_cast<float4*>(L.X + i * RS + c) = lds4(L.X + W.off[i] + c);
    }
    __syncthreads();
    for (int i = tid; i < g.popP; i += kWideThreads) W.off[i] = i * RS;
    __syncthreads();
}

// Inter-task transfer for wide tasks: the candidates are formed in T (row j for candidate j), a
// thread per block of four genes of a half, evaluated, and the accepted ones copied to their
// target rows.
template <int NT, int FUNC>
__device__ __forceinline__ void wide_transfer_in(const EpochArgs& a, const TaskDev& td, const Geo& g, const Lds& L,
                                                 float* T, const Rng& rng, int tid, int nsb) {
    using S = WShape<NT>;
    constexpr int RS = S::RS, HS = S::HS;
    const int k = a.p.transfer_count, TI = a.p.transfer_interval, g0 = a.g0 - td.gen_base;
    const int wave = tid >> 6, lane = tid & 63, col = lane & 31, h = lane >> 5;
    const uint32_t wd = rng.word((uint32_t)g0, P_MIG, 0u, 0u, 0u);
    const int dn = pick_donor(a, (int)rng.task, wd);
    const TaskDev dd = a.tasks[dn];
    const float* mb = a.mailbox + (int64_t)((a.g0 / TI) & 1) * a.mailbox_stride + dd.mb_off;
    const bool same_box = (dd.lo == td.lo && dd.hi == td.hi);
    const float rng_s = td.hi - td.lo, rng_d = dd.hi - dd.lo;
    rank_islands<kWideThreads>(L, g.pop, g.pop, tid);
    __syncthreads();
    const int nu = 2 * nsb;  // blocks of a row
    for (int e = tid; e < k * nu; e += kWideThreads) {
        const int j = e / nu, u = e - j * nu, hh = u >= nsb ? 1 : 0, sb = u - (hh ? nsb : 0);
        const float* mrow = mb + (int64_t)j * dd.dim;
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int d = 2 * (4 * sb + q) + hh;
            v[q] = mrow[d < dd.dim ? d : 0];
        }
        const float4 c4 = lds4(L.X + (int64_t)L.ord[j] * RS + hh * HS + 4 * sb);
        float c[4] = {c4.x, c4.y, c4.z, c4.w};
        U4 ub{0u, 0u, 0u, 0u};
        if (a.p.transfer_cr > 0.0f)
            ub = rng.block((uint32_t)g0, P_XFER, (uint32_t)j, (uint32_t)hh, (uint32_t)sb);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int d = 2 * (4 * sb + q) + hh;
            const bool take = !(a.p.transfer_cr > 0.0f) || uniform01(pick(ub, (uint32_t)q)) > a.p.transfer_cr;
            if (d < g.D && d < dd.dim && take) {
                if (same_box) c[q] = v[q];
                else {
                    const float t1 = v[q] - dd.lo;
                    const float t2 = t1 / rng_d;
                    const float t3 = t2 * rng_s;
                    c[q] = td.lo + t3;
                }
            }
        }
        *reinterpret_cast<float4*>(T + (int64_t)j * RS + hh * HS + 4 * sb) = make_float4(c[0], c[1], c[2], c[3]);
    }
    __syncthreads();
    const int ntc = (k + 31) / 32;
    for (int ct = wave; ct < ntc; ct += kWideThreads / 64) {
        const int j = ct * 32 + col, je = j < k ? j : 0;
        const float f = wide_eval_row<NT, FUNC>(T + (int64_t)je * RS + h * HS, g, L, col, h, nsb);
        if (j < k && h == 0) {
            const int tgt = L.ord[g.pop - k + j];
            const bool acc = f < L.fit[tgt];
            if (acc) L.fit[tgt] = f;
            L.aux[j] = acc ? tgt : -1;
        }
    }
    __syncthreads();
    for (int e = tid; e < k * nu; e += kWideThreads) {
        const int j = e / nu, u = e - j * nu, c = u >= nsb ? HS + 4 * (u - nsb) : 4 * u;
        const int tgt = L.aux[j];
        if (tgt >= 0) *reinterpret_cast<float4*>(L.X + (int64_t)tgt * RS + c) = lds4(T + (int64_t)j * RS + c);
    }
    __syncthreads();
}

// QL: the task's Q image is staged in LDS (the workgroup's first 1024 NT^2 floats) and the
// MFMA A operands come from there instead of L2.
template <int NT, int FUNC, int ALGO, bool QL>
__device__ __forceinline__ void wide_body(const EpochArgs& a, float* smem, const int task, const TaskDev& td) {
    using S = WShape<NT>;
    constexpr int RS = S::RS, HS = S::HS, WT = kWideThreads;
    const int tid = threadIdx.x;
    Geo g;
    g.D = td.dim;
    g.Dh = (g.D + 1) >> 1;
    g.pop = td.pop;
    g.popP = (g.pop + 31) & ~31;
    g.ntiles = g.popP / 32;
    g.m = g.pop / (a.p.n_islands > 0 ? a.p.n_islands : 1);
    g.modD.init((uint32_t)g.D);
    g.modM.init((uint32_t)g.m);
    const int nsb = (g.Dh + 3) >> 2;  // gene blocks per half that hold genes
    Lds L;
    L.X = a.scratch + td.scr_off;
    float* T = L.X + (int64_t)g.popP * RS;
    float* base = smem;
    if constexpr (QL) {
        L.Q = smem;
        base = smem + 1024 * NT * NT;
        // eight 16-byte loads in flight per thread
        const float4* qg = reinterpret_cast<const float4*>(a.Qw + td.qw_off);
        constexpr int n4 = 256 * NT * NT;
        for (int e0 = tid; e0 < n4; e0 += 8 * WT) {
            float4 v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int e = e0 + k * WT;
                v[k] = qg[e < n4 ? e : n4 - 1];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int e = e0 + k * WT;
                if (e < n4) reinterpret_cast<float4*>(smem)[e] = v[k];
            }
        }
    } else {
        L.Q = const_cast<float*>(a.Qw + td.qw_off);
    }
    L.o = base;
    L.tab = L.o + RS;
    L.fit = L.tab + 32 * NT;
    WideLds W;
    W.off = reinterpret_cast<int*>(L.fit + g.popP);
    float* sh = reinterpret_cast<float*>(W.off + g.popP);
    W.mate = reinterpret_cast<int4*>(sh);
    W.jr = reinterpret_cast<int*>(sh + 4 * g.popP);
    W.ps = sh;
    W.pz = sh + 512;
    L.ftmp = sh;
    L.ord = reinterpret_cast<int*>(sh + g.popP);
    L.aux = L.ord + g.popP;
    const Rng rng{a.p.seed_lo, a.p.seed_hi, (uint32_t)task};
    const int lane = tid & 63, col = lane & 31, h = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    for (int e = tid; e < RS + 32 * NT; e += WT) base[e] = 0.0f;
    for (int i = tid; i < g.popP; i += WT) W.off[i] = i * RS;
    __syncthreads();
    for (int d = tid; d < g.D; d += WT) {
        L.o[(d & 1) * HS + (d >> 1)] = a.shift[td.v_off + d];
        L.tab[d] = a.tab[td.v_off + d];
    }
    // rows in the padded layout, zero past the dimension up to the last octet of slots that is read
    const int nblk = 2 * ((g.Dh + 7) >> 3);
    if (a.init) {
        const float lo = td.lo, rng_ = td.hi - td.lo;
        for (int e = tid; e < g.popP * RS; e += WT) {
            const int i = e / RS, c = e - i * RS;
            const int d = (c < HS) ? 2 * c : 2 * (c - HS) + 1;
            float v = 0.0f;
            if (i < g.pop && c < 2 * HS && d < g.D) {
                const float u = uniform01(rng.word(0u, P_INIT, (uint32_t)i, 0u, (uint32_t)d));
                const float t1 = u * rng_;
                v = t1 + lo;
            }
            L.X[e] = v;
        }
    } else {
        stage_rows<RS, HS, WT, 8>(L.X, a.X + td.x_off, g.pop, g.pop, g.D, nblk, tid);
    }
    if (!a.init)
        for (int i = tid; i < g.pop; i += WT) L.fit[i] = a.fit[td.fit_off + i];
    __syncthreads();
    if (a.init) {
        for (int it = wave; it < g.ntiles; it += WT / 64) {
            const int i = it * 32 + col;
            const float f = wide_eval_row<NT, FUNC>(L.X + (int64_t)i * RS + h * HS, g, L, col, h, nsb);
            if (i < g.pop && h == 0) L.fit[i] = f;
        }
        __syncthreads();
    }

    const int TI = a.p.transfer_interval;
    if (transfer_now(a, td)) wide_transfer_in<NT, FUNC>(a, td, g, L, T, rng, tid, nsb);

    const int U = 2 * ((g.Dh + 7) >> 3);  // trial units per individual
    const int ti0 = tid / U, tr0 = tid - ti0 * U;
    const bool islands = a.p.n_islands > 1;
    for (int gen = a.g0 - td.gen_base + 1; gen <= a.g1 - td.gen_base; ++gen) {
        if (islands && a.p.exchange_interval > 0 && gen % a.p.exchange_interval == 0) {
            wide_gather<NT>(g, L, W, tid);
            island_exchange<4 * NT, WT>(a, g, L, T, rng, gen, tid);
        }
        wide_mates<ALGO>(a, g, W, rng, gen, tid);
        __syncthreads();
        wide_trials<NT, ALGO>(a, td, g, L.X, W, rng, gen, ti0, tr0, U);
        __syncthreads();
        // the lane's half index is made opaque (masks derived from it are not hoisted out of
        // the generation loop into spilled scalar registers)
        int hh = h;
        asm volatile("" : "+v"(hh));
        if (g.ntiles > 4) wide_fitness<NT, FUNC, QL>(g, L, W, wave, col, hh, nsb);
        else if (g.ntiles > 2) wide_fitness_split<NT, FUNC, QL, (NT + 1) / 2, 2>(g, L, W, wave, lane, col, hh, nsb);
        else if (g.ntiles > 1) wide_fitness_split<NT, FUNC, QL, (NT + 3) / 4, 4>(g, L, W, wave, lane, col, hh, nsb);
        else wide_fitness_split<NT, FUNC, QL, 1, 8>(g, L, W, wave, lane, col, hh, nsb);
        __syncthreads();
        if (islands && a.p.migrate_interval > 0 && a.p.migrate_count > 0 && gen % a.p.migrate_interval == 0) {
            wide_gather<NT>(g, L, W, tid);
            island_migration<4 * NT, WT>(a, g, L, tid);
        }
    }

    if (a.publish) {
        rank_islands<WT>(L, g.pop, g.pop, tid);
        __syncthreads();
    }
    unstage_rows<HS, WT, 8>(a.X + td.x_off, L.X, [&](int i) { return W.off[i]; }, g.pop, g.D, tid);
    for (int i = tid; i < g.pop; i += WT) a.fit[td.fit_off + i] = L.fit[i];
    if (a.publish) {
        const int k = a.p.transfer_count;
        float* mb = a.mailbox + (int64_t)((a.g1 / TI) & 1) * a.mailbox_stride + td.mb_off;
        for (int e = tid; e < k * g.D; e += WT) {
            const int r = e / g.D, d = e - r * g.D;
            mb[e] = L.X[W.off[L.ord[r]] + (d & 1) * HS + (d >> 1)];
        }
    }
}

// Two waves per SIMD: one workgroup of eight waves a CU at the largest Q images, and at least
// that at the others.
template <int NT, int ALGO, bool QL>
__global__ __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(2))) void wide_epoch_kernel(
    EpochArgs a, const int* __restrict__ order) {
    extern __shared__ __align__(16) float smem[];
    rebase_epoch(a);
    const int task = order[blockIdx.x];
    const TaskDev td = a.tasks[task];
    if (!runs_epoch(a, td)) return;
    switch (td.func) {
    case F_SPHERE: wide_body<NT, F_SPHERE, ALGO, QL>(a, smem, task, td); break;
    case F_ROSENBROCK: wide_body<NT, F_ROSENBROCK, ALGO, QL>(a, smem, task, td); break;
    case F_ACKLEY: wide_body<NT, F_ACKLEY, ALGO, QL>(a, smem, task, td); break;
    case F_RASTRIGIN: wide_body<NT, F_RASTRIGIN, ALGO, QL>(a, smem, task, td); break;
    case F_GRIEWANK: wide_body<NT, F_GRIEWANK, ALGO, QL>(a, smem, task, td); break;
    case F_WEIERSTRASS: wide_body<NT, F_WEIERSTRASS, ALGO, QL>(a, smem, task, td); break;
    case F_SCHWEFEL: wide_body<NT, F_SCHWEFEL, ALGO, QL>(a, smem, task, td); break;
    case F_ELLIPTIC: wide_body<NT, F_ELLIPTIC, ALGO, QL>(a, smem, task, td); break;
    case F_REF_ACKLEY: wide_body<NT, F_REF_ACKLEY, ALGO, QL>(a, smem, task, td); break;
    case F_REF_RASTRIGIN: wide_body<NT, F_REF_RASTRIGIN, ALGO, QL>(a, smem, task, td); break;
    case F_REF_GRIEWANK: case F_REF_GRIEWANK_GA: wide_body<NT, F_REF_GRIEWANK, ALGO, QL>(a, smem, task, td); break;
    case F_REF_WEIERSTRASS: wide_body<NT, F_REF_WEIERSTRASS, ALGO, QL>(a, smem, task, td); break;
    case F_REF_SCHWEFEL: wide_body<NT, F_SCHWEFEL, ALGO, QL>(a, smem, task, td); break;
    default: break;
    }
}
#endif  // EMTF_WIDE_NT

}  // namespace emtf

#if defined(EMTF_WIDE_NT)
#if !defined(EMTF_ALGO)
#error "compile the wide kernel with -DEMTF_WIDE_NT=<row tiles> -DEMTF_ALGO=<0|2>"
#endif
#define EMTF_WCAT(a, b, c, d) a##b##_##c##d
#define EMTF_WNAME(a, b, c, d) EMTF_WCAT(a, b, c, d)

// The Q image in LDS where it fits beside the population's arrays: every population up to
// 1024 for NT <= 5, up to 512 for NT = 6; else read from L2.
static bool wide_q_in_lds(int pop) {
    return EMTF_WIDE_NT <= 6 && 4 * emtf::wide_lds_floats(EMTF_WIDE_NT, pop, true) <= 160 * 1024;
}

extern "C" int EMTF_WNAME(emtf_wide_lds_floats_nt, EMTF_WIDE_NT, a, EMTF_ALGO)(int pop) {
    return emtf::wide_lds_floats(EMTF_WIDE_NT, pop, wide_q_in_lds(pop));
}

template <bool QL>
static hipError_t launch_wide(const emtf::EpochArgs& a, const int* order, int n, int lds_bytes, hipStream_t stream) {
    static bool lds_ok = false;
    auto k = &emtf::wide_epoch_kernel<EMTF_WIDE_NT, EMTF_ALGO, QL>;
    if (!lds_ok) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        lds_ok = true;
    }
    hipLaunchKernelGGL(k, dim3(n), dim3(emtf::kWideThreads), lds_bytes, stream, a, order);
    return hipGetLastError();
}

// lds_bytes: 4 emtf_wide_lds_floats of the unit's largest population, which says whether the Q
// image is in it.
extern "C" int EMTF_WNAME(emtf_launch_wide_nt, EMTF_WIDE_NT, a, EMTF_ALGO)(const emtf::EpochArgs* args, const int* order,
                                                                          int n, int lds_bytes, hipStream_t stream) {
#if EMTF_WIDE_NT <= 6
    if (lds_bytes >= 4 * 1024 * EMTF_WIDE_NT * EMTF_WIDE_NT) return (int)launch_wide<true>(*args, order, n, lds_bytes, stream);
#endif
#if EMTF_WIDE_NT >= 6
    return (int)launch_wide<false>(*args, order, n, lds_bytes, stream);
#else
    return (int)hipErrorInvalidValue;
#endif
}
#else
#if !defined(EMTF_KB) || !defined(EMTF_ALGO)
#error "compile island.hip with -DEMTF_KB=<gene blocks per half> -DEMTF_ALGO=<0|2>"
#endif

#define EMTF_CAT3(a, b, c, d) a##b##_##c##d
#define EMTF_NAME(a, b, c, d) EMTF_CAT3(a, b, c, d)

// emtf_launch_epoch_kb<KB>_a<ALGO>: one instantiation per translation unit.
extern "C" int EMTF_NAME(emtf_launch_epoch_kb, EMTF_KB, a, EMTF_ALGO)(const emtf::EpochArgs* args, const int* order,
                                                                     int n, int lds_bytes, hipStream_t stream) {
    static bool lds_ok = false;
    auto k = &emtf::island_epoch_kernel<EMTF_KB, EMTF_ALGO>;
    if (!lds_ok) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        lds_ok = true;
    }
    hipLaunchKernelGGL(k, dim3(n), dim3(emtf::kThreads), lds_bytes, stream, *args, order);
    return (int)hipGetLastError();
}

// emtf_launch_persist_kb<KB>_a<ALGO>: the persistent schedule's kernel over `blocks`
// workgroups (one per item).
// the kernel's dynamic LDS allowance: 160 KB less its own static LDS (its item slot)
static hipError_t persist_lds_setup() {
    static bool done = false;
    if (done) return hipSuccess;
    const void* k = reinterpret_cast<const void*>(&emtf::island_persistent_kernel<EMTF_KB, EMTF_ALGO>);
    hipFuncAttributes fa{};
    hipError_t e = hipFuncGetAttributes(&fa, k);
    if (e == hipSuccess)
        e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - (int)fa.sharedSizeBytes);
    if (e == hipSuccess) done = true;
    return e;
}

extern "C" int EMTF_NAME(emtf_launch_persist_kb, EMTF_KB, a, EMTF_ALGO)(const emtf::EpochArgs* args,
                                                                       const emtf::PersistArgs* pa, const int* order,
                                                                       int blocks, int lds_bytes, hipStream_t stream) {
    const hipError_t e = persist_lds_setup();
    if (e != hipSuccess) return (int)e;
    auto k = &emtf::island_persistent_kernel<EMTF_KB, EMTF_ALGO>;
    hipLaunchKernelGGL(k, dim3(blocks), dim3(emtf::kThreads), lds_bytes, stream, *args, *pa, order);
    return (int)hipGetLastError();
}


#if EMTF_KB == 2 && EMTF_ALGO == 0
extern "C" int emtf_lds_floats_kb(int pop, int kb) { return emtf::lds_floats_kb(pop, kb); }
extern "C" int emtf_epoch_lds_floats_kb(int pop, int kb) { return emtf::epoch_lds_floats(pop, kb); }
#endif

#if EMTF_ALGO == 0
#define EMTF_OBJ_NAME2(a, b) a##b
#define EMTF_OBJ_NAME(a, b) EMTF_OBJ_NAME2(a, b)

// Polish kernel LDS: Q, o, tab, fit, ord, then the staging of 32 / cpe elite slots.
extern "C" int EMTF_OBJ_NAME(emtf_polish_lds_floats_kb, EMTF_KB)(int pop, int waves, int cpe) {
    using S = emtf::Shape<EMTF_KB>;
    (void)waves;
    const int popP = (pop + 31) & ~31;
    return 32 * S::NT * S::RS + S::RS + 32 * S::NT + 2 * popP + (32 / cpe) * emtf::PolishSlot<EMTF_KB>::floats(cpe) +
           emtf::PolishSlot<EMTF_KB>::kScratch;
}

extern "C" int EMTF_OBJ_NAME(emtf_launch_polish_kb, EMTF_KB)(const emtf::EpochArgs* args, const int* order, int n,
                                                             int lds_bytes, hipStream_t stream) {
    static bool lds_ok = false;
    auto k = &emtf::polish_kernel<EMTF_KB>;
    if (!lds_ok) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        lds_ok = true;
    }
    hipLaunchKernelGGL(k, dim3(n), dim3(emtf::kThreads), lds_bytes, stream, *args, order);
    return (int)hipGetLastError();
}
#endif
#endif  // EMTF_WIDE_NT
