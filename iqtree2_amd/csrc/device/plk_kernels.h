// HIP kernels of the likelihood engine (gfx950, wave64).
//
// Layout in HBM (one instance):
//   partial[slot][p][c][x]   T (double or float), pattern-major, eigen basis;
//                            4 states, and 20 in double storage: as Part says
//   scale[slot][p]           uint16 (FP64 form) / int32 exponent (FP32 form),
//                            [slot][p][c] in safe mode
//   theta[p][c][x]           T; buffer_scale[p] double
//   states[taxon][p]         uint8
// Thread mapping: one thread per (pattern, category); the C threads of a
// pattern are adjacent lanes of one wavefront, so cross-category reductions are
// lane shuffles. The traversals of 4 states (dna_ops) and of 20 in double
// storage (prot_ops) map lanes as their matrix products do. A workgroup owns a
// tile of 256/C patterns and walks the whole post-order op list for that tile:
// patterns are independent, so no synchronisation crosses workgroups.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "plk.h"

namespace plkdev {

constexpr int kThreads = 256;
constexpr double kScaleThreshold64 = 0x1p-256;          // tree/phylotree.h:74-80
constexpr int kScaleExp64 = 256;
constexpr double kLogScaleThreshold = -177.4456782233459932741;
constexpr float kScaleThreshold32 = 0x1p-40f;           // FP32-storage rescale threshold
constexpr double kLn2 = 0.6931471805599453094172321;

// Precision traits: storage type, scale counter type and the rescale rule.
template <typename T> struct Prec;
template <> struct Prec<double> {
    using scale_t = uint16_t;
    // one rescale by 2^256 per underflowing node (tree/phylokernelnew.h:1993-2030)
    __device__ static bool underflow(double m) { return m < kScaleThreshold64; }
    static constexpr double threshold = kScaleThreshold64;   // a block max at or above it never rescales
    __device__ static int exponent(double) { return 1; }
    __device__ static double apply(double v, int) { return ldexp(v, kScaleExp64); }
    // safe mode: a category scaled once more than the least-scaled one is
    // multiplied by 2^-256, more than once is dropped (tree/phylokernelnew.h:2891-2915)
    __device__ static double safe_adjust(int d) {
        return d == 0 ? 1.0 : (d == 1 ? kScaleThreshold64 : 0.0);
    }
    static constexpr double log_unit = kLogScaleThreshold;   // ln(2^-256)
    // an unobserved constant pattern (+ASC): a rescaled one counts once at the
    // scaling threshold, whatever its counter (tree/phylokernelnew.h:2940-2947)
    __device__ static double asc_scale(double v, int minsc) { return minsc != 0 ? v * kScaleThreshold64 : v; }
    __device__ static double asc_scale_log(double v, double bs) { return bs != 0.0 ? v * kScaleThreshold64 : v; }
};
template <> struct Prec<float> {
    using scale_t = int32_t;
    // exact power-of-two rescale that brings the block max into [0.5, 1)
    __device__ static bool underflow(float m) { return m < kScaleThreshold32 && m > 0.0f; }
    static constexpr float threshold = kScaleThreshold32;
    __device__ static int exponent(float m) { return -(ilogbf(m) + 1); }
    __device__ static float apply(float v, int k) { return ldexpf(v, k); }
    // counters are exponents, so categories differ by an exact power of two
    __device__ static double safe_adjust(int d) { return ldexp(1.0, -d); }
    static constexpr double log_unit = -kLn2;
    // counters are exponents: the exact scale back
    __device__ static double asc_scale(double v, int minsc) { return ldexp(v, -minsc); }
    __device__ static double asc_scale_log(double v, double bs) { return v * exp(bs); }
};

struct ModelDev {
    const double* eval;      // [n]
    const double* evec;      // [n][n]
    const double* inv_evec;  // [n][n]
    const double* tip;       // [SU+1][n]
    const double* rates;     // [C]
    const double* props;     // [C]
};

struct InstDev {
    int P, Ppad, n, C, SU, safe;
    const uint8_t* states;   // [ntaxa][Ppad]
    const double* freq;      // [Ppad]
    const double* invar;     // [Ppad]
    void* partial;           // [nslots][Ppad*block]
    void* scale;             // [nslots][Ppad*(safe?C:1)]
    void* theta;             // [Ppad*block]
    double* buffer_scale;    // [Ppad]
    double* ptn_lh;          // [Ppad]
    size_t slot_stride;      // Ppad*block
    size_t scale_stride;     // Ppad*(safe?C:1)
    uint32_t slot_units, scale_units;   // the same in 256 bytes (whole: Ppad is a multiple of 256)
    // +ASC (Lewis): the last nasc of the P patterns are the unobserved
    // constant patterns; pattern k's lh goes to asc[4k], and a derivative
    // evaluation adds lh as the derivative sum counts it, d1 and d2 at 4k+1..3
    int nasc;
    double* asc;
};

// A pointer that was itself read from memory has no address space, and every
// access through it is a flat one (through the LDS aperture check, waiting for
// LDS and memory alike). hbm(p) makes it one to device memory.
template <typename T>
using Hbm = __attribute__((address_space(1))) T;
template <typename T>
__device__ inline T* hbm(T* p) { return (T*)(Hbm<T>*)(uint64_t)p; }
__device__ inline void* hbm(void* p) { return (void*)(Hbm<char>*)(uint64_t)p; }
__device__ inline InstDev on_hbm(InstDev I) {
    I.states = hbm(I.states);
    I.freq = hbm(I.freq);
    I.invar = hbm(I.invar);
    I.partial = hbm(I.partial);
    I.scale = hbm(I.scale);
    I.theta = hbm(I.theta);
    I.buffer_scale = hbm(I.buffer_scale);
    I.ptn_lh = hbm(I.ptn_lh);
    I.asc = hbm(I.asc);
    return I;
}
__device__ inline ModelDev on_hbm(ModelDev m) {
    return ModelDev{hbm(m.eval), hbm(m.evec), hbm(m.inv_evec), hbm(m.tip), hbm(m.rates), hbm(m.props)};
}

// Where slot s keeps value x of (pattern p, category c), element
// at(I, s, p, c) + x(p, x), and its counter, element count_at(I, s, p, c):
// [slot][p], safe mode [slot][p][c]. Values are [slot][p][c][x], but
// 4 states: 64 (pattern, category) pairs, those of 64 / C adjacent patterns,
// make a chunk of 256 values, and in it four patterns' pairs of a category are
// adjacent: pair l = (p / 4, c, p % 4), whose values are
//   float    at 4l + x
//   double   at [g / 2][x][j][g % 2] of pair l = j + 16g (j < 16): a lane's
//            matrix operands, sixteen bytes at a time
// A slot is one stretch of memory, since a sweep reads a slot of all patterns
// at a time: with all slots of a chunk together a pass over the branches of
// 200 taxa x 100,000 sites took 17.2 ms (so: 17.0; float 14.9 and 14.4), and
// the float traversal of 100 x 100,000 took 367 us (so: 357; double 437 both).
// A thread of its own pair reads four values of eight bytes. With two values
// of a pair side by side, and lanes that exchange rows around each load and
// store of dna_ops, the pass took 16.65 ms and an NNI round of it 120 ms (so:
// 123), but one branch's Newton 148 us (144) and small batches 3 to 5% more.
// 20 states in double storage: 32 patterns of a category make a block of 640
// values, the operand registers X = x / 4 of a wavefront's two sixteens S, two
// side by side: [(S0, X0 X1), (S0, X2 X3), the same of S1, (X4, S0 S1)]
// [lane p % 16 + 16 (x % 4)][2], so that a thread of its own (p, c) reads two
// values at a time, too (a sweep of 20 taxa x 1,200 sites with the sixteens
// side by side, one at a time: 2319 us, so: 2150; in [p][c][x] order 2120).
template <typename T, int N, int C>
struct Part {
    static constexpr bool kDna = N == 4, kProt = N == 20 && sizeof(T) == 8, kLanes = kDna && sizeof(T) == 8;
    // (unsigned, so that a thread's place within its tile is worked out once)
    __device__ static size_t at(const InstDev& I, int slot, uint32_t p, uint32_t c) {
        if (kProt) return slot * I.slot_stride + ((size_t)(p >> 5) * C + c) * 640 + (p >> 4 & 1) * 256 + (p & 15) * 2;
        if (!kDna) return slot * I.slot_stride + (size_t)p * (N * C) + c * N;
        const uint32_t l = (p % (64 / C) >> 2) * (4 * C) + 4 * c + (p & 3);
        return (size_t)((uint32_t)slot * I.slot_units) * (256 / sizeof(T)) + (size_t)(p / (64 / C)) * 256 +
               (kLanes ? (l >> 5) * 128 + (l & 15) * 2 + (l >> 4 & 1) : l * 4);
    }
    // value i, from at(), where value 0 is
    __device__ static int x(int p, int i) {
        if (kProt && i < 16) return (i >> 3) * 128 + (i & 3) * 32 + (i >> 2 & 1);
        if (kProt) return 512 - 255 * (p >> 4 & 1) + (i & 3) * 32;
        return kLanes ? 32 * i : i;
    }
    __device__ static size_t count_at(const InstDev& I, int slot, uint32_t p, uint32_t c) {
        if (!kDna) return slot * I.scale_stride + (I.safe ? (size_t)p * C + c : (size_t)p);
        return (size_t)((uint32_t)slot * I.scale_units) * (256 / sizeof(typename Prec<T>::scale_t)) + (I.safe ? p * C + c : p);
    }
};

// Elements of one (op, child) table for 4 states. Double storage: a child's
// matrices, a tip's too (its product with the tip vectors is part of the step,
// dna_ops), as operands of the matrix products: lane l's elements of a step,
// child 0's then child 1's, are adjacent (dna_frag). Float storage: an internal
// child's matrices [C][4][4], a tip child's lookup [SU+1][C][4], whose product
// is rounded once.
__host__ __device__ inline int dna_table_size(int C, int SU, size_t elem) {
    const int mat = C == 8 ? 128 : 64, lut = (SU + 1) * C * 4;
    return elem == 8 ? mat : lut > C * 16 ? lut : C * 16;
}
// where element (x, i) of category c's matrix of child k goes among a step's
// 2 * dna_table_size elements: f(place) for each copy
template <typename F>
__device__ inline void dna_frag(int C, int c, int x, int i, int k, F f) {
    for (int b = 0; b < 4; b++)
        for (int h = 0; h < (C == 8 ? 2 : 1); h++) {
            const int cat = C == 1 ? 0 : C == 2 ? b & 1 : C == 4 ? b : b + 4 * h;
            if (cat == c) f(128 * h + 2 * (x + 4 * b + 16 * i) + k);
        }
}

// Transition tables of protein (20-state) internal children are stored in
// the operand order of the matrix-core tile (plk_mfma.h).
constexpr int kProtN = 20;                 // protein states
constexpr int kProtKSteps = 5;             // 4-wide K steps over 20 states
constexpr int kProtFrag = 2 * kProtKSteps * 64;   // fragment elements per category

// Elements of one (op, child) table for 20 states. Float storage: an internal
// child in fragment order (C categories), a tip child's lookup [SU+1][C][20].
// Double storage: a step's are [C][2 children][kProtKid], an internal child's
// matrix as 4x4 blocks (prot_ops), a tip child's lookup [SU+1][20], or its
// matrix if the lookup is larger than kProtKid.
constexpr int kProtBlocks = 13 * 32;      // 25 blocks of 16, in pairs
constexpr int kProtKid = 512;
__host__ __device__ inline bool prot_lut(int SU) { return (SU + 1) * kProtN <= kProtKid; }
__host__ __device__ inline int prot_table_size(int C, int SU, size_t elem) {
    const int frag = C * kProtFrag, lut = (SU + 1) * C * kProtN;
    return elem == 8 ? C * kProtKid : frag > lut ? frag : lut;
}
// A 20x20 matrix as blocks B of 4x4, each two at [B / 2][x % 4 + 4 (k % 4)][B % 2],
// in the order in which prot_ops multiplies: the rows X = x / 4 two at a time
// along K = k / 4, then the fifth. The (x, k) of element t, x = -1 past the last.
__host__ __device__ inline void prot_block_index(int t, int& x, int& k) {
    const int B = 2 * (t >> 5) + (t & 1), e = t >> 1 & 15;
    const int X = B >= 20 ? 4 : B / 10 * 2 + B % 2, K = B >= 20 ? B - 20 : B % 10 / 2;
    x = B < 25 ? 4 * X + (e & 3) : -1;
    k = 4 * K + (e >> 2);
}

// Fragment order of an internal child's table, per category:
// frag[xb][st][lane] = E[x = 16 xb + lane % 16][k = 5 (lane / 16) + st],
// zero for x >= 20. Returns the (x, k) of element t, x = -1 for padding.
__host__ __device__ inline void prot_frag_index(int t, int& x, int& k) {
    const int xb = t / (kProtKSteps * 64), st = (t / 64) % kProtKSteps, l = t & 63;
    x = 16 * xb + (l & 15);
    k = 5 * (l >> 4) + st;
    if (x >= kProtN) x = -1;
}

// A plain device copy of a known size (each launch reads and writes n*32
// bytes): the HBM bandwidth a streaming kernel reaches, and the reference
// size that calibrates the hardware byte counters.
__global__ void __launch_bounds__(kThreads)
k_copy(const double4* __restrict__ src, double4* __restrict__ dst, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

enum TraverseMode { MODE_PARTIALS = 0, MODE_BRANCH = 1, MODE_THETA = 2 };
enum BufferMode { BUF_DERV = 0, BUF_LNL = 1 };

// One traversal step for dna_ops and prot_ops: scalar loads of sixteen bytes,
// each made when its part of the step is due.
struct alignas(64) TileOp {
    uint64_t tip[2];      // a tip child's row of states (others: taxon 0's)
    uint32_t v[2], sc[2]; // where a slot child's values and counters begin, kNoSlot for one that comes from elsewhere
    uint32_t dst, dsc;    // the dad's; in units of 256 bytes from slot 0, so that 32 bits reach 1 TB (20 states: slots)
    uint32_t kind;        // of child k in bits 2k and 2k + 1, below
    uint32_t root;        // bit k: child k is the root leaf (state-basis models)
};
// a slot in memory, the dad of the step before (in registers), the dad of the
// step before that, a tip
enum TileChild { CHILD_SLOT = 0, CHILD_LAST = 1, CHILD_LAST2 = 2, CHILD_TIP = 3 };
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;
constexpr int kTileAhead = 6;                // steps that dna_ops looks ahead: copies of the last TileOp

// steps nops .. nops + kTileAhead - 1 repeat the last
__device__ inline void make_tile_op(const InstDev& I, const plk_op* __restrict__ ops, int o, int nops, TileOp* tops,
                                    unsigned root = 0) {
    const plk_op op = ops[o];
    const int last = o > 0 ? ops[o - 1].dad_slot : -1, last2 = o > 1 ? ops[o - 2].dad_slot : -1;
    const uint32_t nv = I.n != 4 ? 1 : I.slot_units, nc = I.n != 4 ? 1 : I.scale_units;
    TileOp t;
    t.kind = 0;
    for (int k = 0; k < 2; k++) {
        const int id = op.child[k].id;
        const int kind = op.child[k].is_tip ? CHILD_TIP : id == last ? CHILD_LAST : id == last2 && I.n == 4 ? CHILD_LAST2 : CHILD_SLOT;
        t.kind |= kind << 2 * k;
        t.tip[k] = reinterpret_cast<uint64_t>(I.states) + (kind == CHILD_TIP ? (size_t)id * I.Ppad : 0);
        t.v[k] = kind == CHILD_SLOT ? id * nv : kNoSlot;
        t.sc[k] = kind == CHILD_SLOT ? id * nc : kNoSlot;
    }
    t.dst = op.dad_slot * nv;
    t.dsc = op.dad_slot * nc;
    t.root = root;
    tops[o] = t;
    if (o == nops - 1)
        for (int a = 1; a <= kTileAhead; a++) tops[o + a] = t;
}

// ---------------------------------------------------------------------------
// computePartialInfo (tree/phylokernelnew.h:1008-1109): per op and child, the
// eigen-basis transition rows echild[c][x][i] = evec[x][i] exp(eval[i] r_c t)
// for an internal child, or the tip table leaf[s][c][x] =
// sum_i echild[c][x][i] tip[s][i] (leaf[SU] = 1) for a tip child.
// One workgroup per (op, child, category); tables are written in storage
// precision. 4 states, and 20 in double storage: also the steps' TileOps.
template <typename T>
__global__ void __launch_bounds__(kThreads)
k_prep_ops(const plk_op* __restrict__ ops, int nops, ModelDev m, int n, int C, int SU,
           int table_size, T* __restrict__ tables, InstDev I, TileOp* __restrict__ tops) {
    // one block per (op, child, category); LDS: ex[n], then for a tip child
    // U[n][n] and the tip vectors [SU][n]
    extern __shared__ double sh[];
    const int o = blockIdx.x >> 1, k = blockIdx.x & 1, c = blockIdx.y;
    if (o >= nops) return;
    if (tops && k == 0 && c == 0 && threadIdx.x == 0) make_tile_op(I, ops, o, nops, tops);
    const plk_child ch = ops[o].child[k];
    double* ex = sh;
    for (int i = threadIdx.x; i < n; i += blockDim.x) ex[i] = exp(m.eval[i] * (m.rates[c] * ch.length));
    T* out = tables + (size_t)(2 * o + k) * table_size;
    T* kid = tables + (size_t)2 * o * table_size + (2 * c + k) * kProtKid;   // 20 states, double storage
    const bool tip_matrix = sizeof(T) == 8 && (n == 4 || (n == kProtN && !prot_lut(SU)));
    if (!ch.is_tip || tip_matrix) {
        __syncthreads();
        if (n == kProtN && sizeof(T) == 8) {
            for (int t = threadIdx.x; t < kProtBlocks; t += blockDim.x) {
                int x, i;
                prot_block_index(t, x, i);
                kid[t] = x < 0 ? (T)0 : (T)(m.evec[x * n + i] * ex[i]);
            }
            return;
        }
        if (n == kProtN) {
            // the matrix-core tile's fragment order
            T* oc = out + (size_t)c * kProtFrag;
            for (int t = threadIdx.x; t < kProtFrag; t += blockDim.x) {
                int x, i;
                prot_frag_index(t, x, i);
                oc[t] = x < 0 ? (T)0 : (T)(m.evec[x * n + i] * ex[i]);
            }
            return;
        }
        if (n == 4 && sizeof(T) == 8) {
            T* step = tables + (size_t)2 * o * table_size;
            for (int t = threadIdx.x; t < 16; t += blockDim.x) {
                const T v = (T)(m.evec[t] * ex[t % 4]);
                dna_frag(C, c, t / 4, t % 4, k, [&](int at) { step[at] = v; });
            }
            return;
        }
        T* oc = out + (size_t)c * n * n;
        for (int t = threadIdx.x; t < n * n; t += blockDim.x) {
            const int i = t % n, x = t / n;
            oc[t] = (T)(m.evec[x * n + i] * ex[i]);
        }
        return;
    }
    double* ev_sh = ex + n;
    double* tp_sh = ev_sh + n * n;
    for (int t = threadIdx.x; t < n * n; t += blockDim.x) ev_sh[t] = m.evec[t];
    for (int t = threadIdx.x; t < SU * n; t += blockDim.x) tp_sh[t] = m.tip[t];
    __syncthreads();
    for (int t = threadIdx.x; t < (SU + 1) * n; t += blockDim.x) {
        const int x = t % n, s = t / n;
        double v;
        if (s == SU) {
            v = 1.0;
        } else {
            const double* ev = ev_sh + x * n;
            const double* tp = tp_sh + s * n;
            v = ev[0] * ex[0] * tp[0];
            for (int i = 1; i < n; i++) v += ev[i] * ex[i] * tp[i];
        }
        if (n == kProtN && sizeof(T) == 8) kid[t] = (T)v;
        else out[(size_t)(s * C + c) * n + x] = (T)v;
    }
}

// Root tables for the branch likelihood (tree/phylokernelnew.h:2713-2806):
// val[c][i] = exp(eval[i] r_c t) p_c, and for a tip dad
// lut[s][c][i] = val[c][i] * tip[s][i] for every s in 0..SU.
__global__ void __launch_bounds__(kThreads)
k_prep_root(ModelDev m, int n, int C, int SU, double length, int tip_dad, double* __restrict__ out) {
    const int nv = C * n;
    for (int t = threadIdx.x; t < nv; t += blockDim.x) {
        const int c = t / n, i = t % n;
        out[t] = exp(m.eval[i] * (m.rates[c] * length)) * m.props[c];
    }
    if (!tip_dad) return;
    const int total = (SU + 1) * nv;
    for (int t = threadIdx.x; t < total; t += blockDim.x) {
        const int i = t % n, c = (t / n) % C, s = t / nv;
        out[nv + t] = exp(m.eval[i] * (m.rates[c] * length)) * m.props[c] * m.tip[s * n + i];
    }
}

// ---------------------------------------------------------------------------
// A pattern's C category values sit in C adjacent lanes (C = 1, 2, 4, 8).
// lane_get<C, K>(v): the value of lane K of this lane's group. For C <= 4 the
// group lies inside one quad and a DPP quad permutation moves the value (no
// LDS round trip); 8 lanes use a bpermute.
template <int C, int K>
__device__ inline int lane_get_i32(int v) {
    if constexpr (C == 1) {
        return v;
    } else if constexpr (C <= 4) {
        constexpr int a = K, b = C == 4 ? K : 2 + K;   // C = 2: lanes {0,1} and {2,3}
        constexpr int ctrl = a | (a << 2) | (b << 4) | (b << 6);
        return __builtin_amdgcn_update_dpp(0, v, ctrl, 0xf, 0xf, false);
    } else {
        const int base = (threadIdx.x & 63) & ~(C - 1);
        return __shfl(v, base + K);
    }
}
template <int C, int K>
__device__ inline double lane_get(double v) {
    const long long x = __double_as_longlong(v);
    const int lo = lane_get_i32<C, K>((int)(unsigned)(x & 0xffffffffll));
    const int hi = lane_get_i32<C, K>((int)(x >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
// max over the 16 lanes of this lane's DPP row (every lane gets it): quad
// swaps, then half-row and row mirrors pair each quad with the others
template <int CTRL>
__device__ inline float dpp_f32(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ inline double dpp_f64(double v) {
    const long long x = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(x & 0xffffffffll), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
template <int CTRL>
__device__ inline float dpp_move(float v) { return dpp_f32<CTRL>(v); }
template <int CTRL>
__device__ inline double dpp_move(double v) { return dpp_f64<CTRL>(v); }
template <typename T>
__device__ inline T row16_max(T m) {
    m = fmax(m, dpp_move<0xB1>(m));    // quad_perm [1,0,3,2]
    m = fmax(m, dpp_move<0x4E>(m));    // quad_perm [2,3,0,1]
    m = fmax(m, dpp_move<0x141>(m));   // row_half_mirror
    m = fmax(m, dpp_move<0x140>(m));   // row_mirror
    return m;
}

// the C values of this lane's group, in category order
template <int C, int K = 0>
__device__ inline void lane_gather(double v, double* out) {
    if constexpr (K < C) {
        out[K] = lane_get<C, K>(v);
        lane_gather<C, K + 1>(v, out);
    }
}

template <int C>
__device__ inline double group_max(double v) {
    double vals[C];
    lane_gather<C>(v, vals);
    double m = vals[0];
#pragma unroll
    for (int c = 1; c < C; c++) m = fmax(m, vals[c]);
    return m;
}
template <int C, int K = 0>
__device__ inline int group_min_int(int v) {
    if constexpr (K + 1 < C) return min(lane_get_i32<C, K>(v), group_min_int<C, K + 1>(v));
    else return lane_get_i32<C, K>(v);
}
// sum over the C lanes of a pattern in category order 0..C-1 (the order the
// reference accumulates lh_cat), result in every lane of the group
template <int C>
__device__ inline double group_sum_ordered(double v) {
    double vals[C];
    lane_gather<C>(v, vals);
    double s = vals[0];
#pragma unroll
    for (int c = 1; c < C; c++) s += vals[c];
    return s;
}
// sumVec<VectorClass, true> grouping over categories (tree/phylokernelnew.h:43-71)
template <int C>
__device__ inline double group_sum_sumvec(double v) {
    double vals[C];
    lane_gather<C>(v, vals);
    double x = 0.0;
    constexpr int cruft = C & 3;
    if (cruft < C) {
        double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
#pragma unroll
        for (int c = 0; c < C - cruft; c += 4) {
            a0 += vals[c]; a1 += vals[c + 1]; a2 += vals[c + 2]; a3 += vals[c + 3];
        }
        a0 += a2;
        a1 += a3;
        a0 += a1;
        x += a0;
    }
#pragma unroll
    for (int c = C - cruft; c < C; c++) x += vals[c];
    return x;
}

// Sum over the 64 lanes of a wavefront with the same bits in every lane:
// DPP quad swaps and row mirrors (each step adds the same two operands in
// both partner lanes) give every lane its 16-lane row sum, then the four row
// sums are read as scalars and added in a fixed order.
__device__ inline double wave_sum(double v) {
    v += dpp_f64<0xB1>(v);    // quad_perm [1,0,3,2]
    v += dpp_f64<0x4E>(v);    // quad_perm [2,3,0,1]
    v += dpp_f64<0x141>(v);   // row_half_mirror
    v += dpp_f64<0x140>(v);   // row_mirror
    const long long x = __double_as_longlong(v);
    const int lo = (int)(unsigned)(x & 0xffffffffll), hi = (int)(x >> 32);
    double r[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const unsigned l = (unsigned)__builtin_amdgcn_readlane(lo, 16 * k);
        const unsigned h = (unsigned)__builtin_amdgcn_readlane(hi, 16 * k);
        r[k] = __longlong_as_double((long long)(((unsigned long long)h << 32) | l));
    }
    return (r[0] + r[1]) + (r[2] + r[3]);
}

// Deterministic workgroup sum: wave_sum inside each wavefront, then the
// wavefront partials in index order. Result valid in thread 0. GUARD = false
// skips the barrier that protects sh from a previous reader, for callers
// whose last use of sh already ended with a barrier.
template <int NV, bool GUARD = true>
__device__ inline void block_sum(double (&v)[NV], double* sh) {
#pragma unroll
    for (int j = 0; j < NV; j++) v[j] = wave_sum(v[j]);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (GUARD) __syncthreads();
    if (lane == 0)
#pragma unroll
        for (int j = 0; j < NV; j++) sh[wave * NV + j] = v[j];
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = blockDim.x >> 6;
#pragma unroll
        for (int j = 0; j < NV; j++) {
            double s = sh[j];
            for (int w = 1; w < nw; w++) s += sh[w * NV + j];
            v[j] = s;
        }
    }
}

// ---------------------------------------------------------------------------
// One binary traversal step for the pattern/category (p, c) of this thread
// (computePartialLikelihoodSIMD, tree/phylokernelnew.h:1632-2031):
// tmp[x] = prod_children (tip: leaf[s][c][x]; internal: sum_i E[c][x][i] child[i]),
// dad = U^-1 tmp, then the reference's rescaling rule. tL / tR are the
// children's tables (tip lookup or transition rows), a tip child goes left.
// Split into the loads (op_load) and the arithmetic and stores (op_finish)
// so that a caller can have the loads of several patterns in flight.
template <typename T, int N>
struct OpIn {
    T l[N], r[N];   // internal children's partials (unused for a tip child)
    int sl, sr;     // tip children's states
    int scl, scr;   // internal children's scale counters
};

template <typename T, int N, int C>
__device__ inline void op_load(const InstDev& I, int l_tip, int l_id, int r_tip, int r_id, int p, int c,
                               OpIn<T, N>& in) {
    using ST = typename Prec<T>::scale_t;
    const T* partial = reinterpret_cast<const T*>(I.partial);
    const ST* scale = reinterpret_cast<const ST*>(I.scale);
    in.scl = in.scr = 0;
    if (l_tip) {
        in.sl = I.states[(size_t)l_id * I.Ppad + p];
    } else {
        const T* src = partial + Part<T, N, C>::at(I, l_id, p, c);
#pragma unroll
        for (int i = 0; i < N; i++) in.l[i] = src[Part<T, N, C>::x(p, i)];
        in.scl = scale[Part<T, N, C>::count_at(I, l_id, p, c)];
    }
    if (r_tip) {
        in.sr = I.states[(size_t)r_id * I.Ppad + p];
    } else {
        const T* src = partial + Part<T, N, C>::at(I, r_id, p, c);
#pragma unroll
        for (int i = 0; i < N; i++) in.r[i] = src[Part<T, N, C>::x(p, i)];
        in.scr = scale[Part<T, N, C>::count_at(I, r_id, p, c)];
    }
}

template <typename T, int N, int C>
__device__ inline void op_finish(const InstDev& I, const T* inv_sh, const T* tL, const T* tR, int l_tip,
                                 int r_tip, int dad_slot, int p, int c, const OpIn<T, N>& in) {
    using ST = typename Prec<T>::scale_t;
    T* partial = reinterpret_cast<T*>(I.partial);
    ST* scale = reinterpret_cast<ST*>(I.scale);
    const bool safe = I.safe != 0;
    T tmp[N];
    if (l_tip) {
        const T* lut = tL + (in.sl * C + c) * N;
#pragma unroll
        for (int x = 0; x < N; x++) tmp[x] = lut[x];
    } else {
        const T* E = tL + c * N * N;
#pragma unroll
        for (int x = 0; x < N; x++) {
            T acc = E[x * N] * in.l[0];
#pragma unroll
            for (int i = 1; i < N; i++) acc = fma(E[x * N + i], in.l[i], acc);
            tmp[x] = acc;
        }
    }
    if (r_tip) {
        const T* lut = tR + (in.sr * C + c) * N;
#pragma unroll
        for (int x = 0; x < N; x++) tmp[x] *= lut[x];
    } else {
        const T* E = tR + c * N * N;
#pragma unroll
        for (int x = 0; x < N; x++) {
            T acc = E[x * N] * in.r[0];
#pragma unroll
            for (int i = 1; i < N; i++) acc = fma(E[x * N + i], in.r[i], acc);
            tmp[x] *= acc;
        }
    }
    // back to the eigen basis: dad[i] = sum_x inv_evec[i][x] tmp[x]
    T dadv[N];
    T lmax = (T)0;
#pragma unroll
    for (int i = 0; i < N; i++) {
        T acc = inv_sh[i * N] * tmp[0];
#pragma unroll
        for (int x = 1; x < N; x++) acc = fma(inv_sh[i * N + x], tmp[x], acc);
        dadv[i] = acc;
        lmax = fmax(lmax, fabs(acc));
    }
    int sc = in.scl + in.scr;
    if (!(l_tip && r_tip)) {   // tip-tip steps are never rescaled
        const bool no_invar = I.invar[p] == 0.0;
        const T m = safe ? lmax : (T)group_max<C>((double)lmax);
        if (Prec<T>::underflow(m) && no_invar) {
            const int k = Prec<T>::exponent(m);
#pragma unroll
            for (int i = 0; i < N; i++) dadv[i] = Prec<T>::apply(dadv[i], k);
            sc += k;
        }
    }
    T* dst = partial + Part<T, N, C>::at(I, dad_slot, p, c);
#pragma unroll
    for (int i = 0; i < N; i++) dst[Part<T, N, C>::x(p, i)] = dadv[i];
    if (safe || c == 0) scale[Part<T, N, C>::count_at(I, dad_slot, p, c)] = (ST)sc;
}

template <typename T, int N, int C>
__device__ inline void op_apply(const InstDev& I, const T* inv_sh, const T* tL, const T* tR,
                                int l_tip, int l_id, int r_tip, int r_id, int dad_slot, int p,
                                int c) {
    OpIn<T, N> in;
    op_load<T, N, C>(I, l_tip, l_id, r_tip, r_id, p, c, in);
    op_finish<T, N, C>(I, inv_sh, tL, tR, l_tip, r_tip, dad_slot, p, c, in);
}

// ---------------------------------------------------------------------------
// A whole op list for a wavefront's 64 (pattern, category) pairs, 4 states,
// on the matrix cores. The same sums in the same order as op_finish: the 4x4
// products are exact chains of fused multiply-adds.
//
// What bounds a step: with tables and children read through LDS and memory, a
// step of a small tree took 2.0 us (two barriers, the tables' trip to LDS, the
// dad's values back from L2), and its matrix rows took 384 bytes of LDS reads
// a thread. A 4x4x4 product of four blocks takes one matrix element a lane
// instead, its result is laid out as its operand, and so are the slots (Part):
// a step is the children's products, their elementwise product and U^-1. No
// barrier, no shuffle; a tip's vectors come from LDS, where they stay. A large
// tree is bound by the vector memory path of its CU (16 bytes of a lane a
// cycle and quad), so
//   - the last two dads' values and counters stay in registers. In post-order
//     every step but a cherry has the last one as a child: of a random tree's
//     child reads a fifth remains;
//   - what a step reads is loaded two steps ahead. Loads and stores share one
//     in-order counter, so a wait for a load is one for all before it, but not
//     for the stores of the two steps since;
//   - a step makes few accesses: both children's matrices in one, the tips'
//     states through the scalar cache, and slots only of children that are read.
// Measured, whole kernel, 198 steps: 1,000 patterns 136 us, 100,000
// 695 us in double (2.6 GB written), the kernel of a thread a pair,
// with tables in LDS, 415 and 1,153.
typedef unsigned tile_u4 __attribute__((ext_vector_type(4)));
using Buffer = __amdgpu_buffer_rsrc_t;

// `bytes` from `base` on; reads past them give 0
__device__ inline Buffer buffer_of(uint64_t base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000);
}

// the constant address space: a scalar load, whatever was stored before
__device__ inline tile_u4 load_u4(uint64_t p) { return *(const __attribute__((address_space(4))) tile_u4*)p; }

// The pairs of a wavefront, in the order of Part: pair j + 4b + 16g is lane
// j + 4b + 16g's own (its state, its counter). The four pairs of a (b, g)
// share a category, as a block of the matrix products does.
template <int C>
struct Pairs {
    static constexpr int kPatterns = 64 / C;
    __device__ static int cat(int b, int g) { return C == 1 ? 0 : C == 2 ? b & 1 : C == 4 ? b : b + 4 * (g & 1); }
    __device__ static int cat(int lane) { return cat(lane >> 2 & 3, lane >> 4); }
    __device__ static int pattern(int lane) {
        const int j = lane & 3, b = lane >> 2 & 3, g = lane >> 4;
        return C == 1 ? lane : C == 2 ? j + 4 * (b >> 1) + 8 * g : C == 4 ? j + 4 * g : j + 4 * (g >> 1);
    }
    // the pairs of pair 0's pattern; those of pair l's: kMask << (l & ~kBits)
    static constexpr unsigned long long kMask = C == 1 ? 0x1ull : C == 2 ? 0x11ull : C == 4 ? 0x1111ull : 0x11111111ull;
    static constexpr int kBits = 4 * (C - 1);
};

// 4x4 matrices times a wavefront's 4-vectors, four registers a lane:
//   double  v_mfma_f64_4x4x4: four blocks of 4x4 by 4x4. A[i][k] of block b in
//           lane i + 4b + 16k; B and D alike, D[i][j] in lane j + 4b + 16i. So
//           register g of lane j + 4b + 16x holds value x of pair j + 4b + 16g
//   float   v_mfma_f32_4x4x1: sixteen blocks, four steps of k. Register x of
//           lane l holds value x of pair l
template <typename T, int C> struct Mat4;
template <int C> struct Mat4<double, C> {
    static constexpr int kA = C == 8 ? 2 : 1;   // matrices of the even and odd registers
    struct A {
        double v[kA];
    };
    // both children's elements of a step (dna_frag); the same matrix M in every block
    __device__ static void load(const Hbm<double>* step, int, int lane, A (&e)[2]) {
        typedef double d2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int h = 0; h < kA; h++) {
            const d2 w = ((const Hbm<d2>*)step)[64 * h + lane];
            e[0].v[h] = w[0];
            e[1].v[h] = w[1];
        }
    }
    __device__ static A load_same(const double* M, int lane) {
        A a;
#pragma unroll
        for (int h = 0; h < kA; h++) a.v[h] = M[(lane & 3) * 4 + (lane >> 4)];
        return a;
    }
    __device__ static void mul(const A& a, const double (&b)[4], double (&d)[4]) {
#pragma unroll
        for (int g = 0; g < 4; g++) d[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.v[g % kA], b[g], 0.0, 0, 0, 0);
    }
    static constexpr int kRow = 1;              // a tip's row of its lookup: none, its vectors wait in LDS
    // the states of a wavefront's patterns, in scalar registers where a
    // register's pairs have theirs in one word of them (a vector load of single
    // bytes takes the memory path as long as one of a kilobyte)
    static constexpr bool kWords = C >= 4;
    static constexpr int kStates = kWords ? 16 / C : 1;
    __device__ static void load_slot(Buffer r, uint32_t at, double (&v)[4]) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const tile_u4 w = __builtin_amdgcn_raw_buffer_load_b128(r, at + 1024 * h, 0, 0);
#pragma unroll
            for (int m = 0; m < 2; m++)
                v[2 * h + m] = __longlong_as_double((long long)((unsigned long long)w[2 * m + 1] << 32 | w[2 * m]));
        }
    }
    __device__ static void store_slot(Buffer r, uint32_t at, const double (&d)[4]) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            tile_u4 w;
#pragma unroll
            for (int m = 0; m < 2; m++) {
                const unsigned long long u = (unsigned long long)__double_as_longlong(d[2 * h + m]);
                w[2 * m] = (unsigned)u;
                w[2 * m + 1] = (unsigned)(u >> 32);
            }
            __builtin_amdgcn_raw_buffer_store_b128(w, r, at + 1024 * h, 0, 0);
        }
    }
    __device__ static void load_row(const Hbm<double>*, bool, int, int, double (&)[kRow]) {}
    // a tip's product: its matrices times the tip vectors (the root leaf's: times 1, 0, 0, 0),
    // 1 for the unknown state su
    __device__ static void tip(const A& a, const double (&)[kRow], const unsigned (&st)[kStates], bool root,
                               const double* tip_sh, int su, int lane, double (&f)[4]) {
        int s[4];
        if constexpr (kWords) {
#pragma unroll
            for (int g = 0; g < 4; g++) s[g] = st[C == 4 ? g : g >> 1] >> 8 * (lane & 3) & 0xff;
        } else {
            // row g of lanes holds the states of register g's pairs: each to every row
            const auto w = __builtin_amdgcn_permlane32_swap(st[0], st[0], false, false);
            const auto lo = __builtin_amdgcn_permlane16_swap(w[0], w[0], false, false);
            const auto hi = __builtin_amdgcn_permlane16_swap(w[1], w[1], false, false);
            s[0] = lo[0];
            s[1] = lo[1];
            s[2] = hi[0];
            s[3] = hi[1];
        }
        double b[4];
        if (root) {
#pragma unroll
            for (int g = 0; g < 4; g++) b[g] = lane < 16 ? 1.0 : 0.0;
            su = -1;
        } else {
#pragma unroll
            for (int g = 0; g < 4; g++) b[g] = tip_sh[s[g] * 4 + (lane >> 4)];
        }
        mul(a, b, f);
        unsigned long long any = 0;
#pragma unroll
        for (int g = 0; g < 4; g++) any |= __builtin_amdgcn_ballot_w64(s[g] == su);
        if (any)
#pragma unroll
            for (int g = 0; g < 4; g++) f[g] = s[g] == su ? 1.0 : f[g];
    }
    // pairs with every value below the threshold, as a mask
    __device__ static unsigned long long small(const double (&d)[4]) {
        unsigned long long m[4], any = 0;
#pragma unroll
        for (int g = 0; g < 4; g++) any |= m[g] = __builtin_amdgcn_ballot_w64(fabs(d[g]) < Prec<double>::threshold);
        if (!any) return 0;
        unsigned long long out = 0;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            m[g] &= m[g] >> 32;
            m[g] &= m[g] >> 16;
            out |= (m[g] & 0xffff) << 16 * g;
        }
        return out;
    }
    // rescale the pairs for which `mine` holds; what their counters gain
    template <bool>
    __device__ static int rescale(double (&d)[4], bool mine, int lane) {
        const unsigned long long m = __builtin_amdgcn_ballot_w64(mine);
#pragma unroll
        for (int g = 0; g < 4; g++)
            if (m >> (16 * g + (lane & 15)) & 1) d[g] = Prec<double>::apply(d[g], 1);
        return mine ? 1 : 0;
    }
};
template <int C> struct Mat4<float, C> {
    typedef float f4 __attribute__((ext_vector_type(4)));
    struct A {
        float v[4];
    };
    // rows of both children's E[c][x][i]
    __device__ static void load(const Hbm<float>* step, int table_size, int lane, A (&e)[2]) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const f4 w = *(const Hbm<f4>*)(step + c * table_size + Pairs<C>::cat(lane) * 16 + (lane & 3) * 4);
#pragma unroll
            for (int k = 0; k < 4; k++) e[c].v[k] = w[k];
        }
    }
    __device__ static A load_same(const double* M, int lane) {
        A a;
#pragma unroll
        for (int k = 0; k < 4; k++) a.v[k] = (float)M[(lane & 3) * 4 + k];
        return a;
    }
    __device__ static void mul(const A& a, const float (&b)[4], float (&d)[4]) {
        f4 acc = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 4; k++) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a.v[k], b[k], acc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; r++) d[r] = acc[r];
    }
    static constexpr int kRow = 4;
    static constexpr bool kWords = false;
    static constexpr int kStates = 1;
    __device__ static void load_slot(Buffer r, uint32_t at, float (&v)[4]) {
        const tile_u4 w = __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0);
#pragma unroll
        for (int x = 0; x < 4; x++) v[x] = __uint_as_float(w[x]);
    }
    __device__ static void store_slot(Buffer r, uint32_t at, const float (&d)[4]) {
        tile_u4 w;
#pragma unroll
        for (int x = 0; x < 4; x++) w[x] = __float_as_uint(d[x]);
        __builtin_amdgcn_raw_buffer_store_b128(w, r, at, 0, 0);
    }
    // a tip's row of its lookup [SU+1][C][4] (others: the first)
    __device__ static void load_row(const Hbm<float>* table, bool tip, int st, int lane, float (&row)[kRow]) {
        const f4 w = *(const Hbm<f4>*)(table + (tip ? (st * C + Pairs<C>::cat(lane)) * 4 : 0));
#pragma unroll
        for (int x = 0; x < 4; x++) row[x] = w[x];
    }
    __device__ static void tip(const A&, const float (&row)[kRow], const unsigned (&)[kStates], bool, const double*, int,
                               int, float (&f)[4]) {
#pragma unroll
        for (int x = 0; x < 4; x++) f[x] = row[x];
    }
    __device__ static float top(const float (&d)[4]) {
        return fmax(fmax(fabs(d[0]), fabs(d[1])), fmax(fabs(d[2]), fabs(d[3])));
    }
    __device__ static unsigned long long small(const float (&d)[4]) {
        return __builtin_amdgcn_ballot_w64(top(d) < Prec<float>::threshold);
    }
    // by the power of two that brings the pattern's (safe: the pair's) maximum into [0.5, 1)
    template <bool kSafe>
    __device__ static int rescale(float (&d)[4], bool mine, int lane) {
        float m = top(d);
        if (!kSafe)
#pragma unroll
            for (int w = 4; w < 4 * C; w <<= 1) m = fmax(m, __shfl_xor(m, w));
        if (!mine || !Prec<float>::underflow(m)) return 0;
        const int k = Prec<float>::exponent(m);
#pragma unroll
        for (int x = 0; x < 4; x++) d[x] = Prec<float>::apply(d[x], k);
        return k;
    }
};

// LDS of dna_ops: the tip vectors
__host__ __device__ inline size_t dna_ops_smem(int SU) { return (size_t)(SU + 1) * 4 * sizeof(double); }

// p_first: the workgroup's first of 256 / C patterns (uniform). tip_sh:
// dna_ops_smem(SU).
template <typename T, int C>
__device__ inline void dna_ops(const InstDev& I, const ModelDev& m, const TileOp* tops, int nops, const T* tables_g,
                               int table_size, int p_first, double* tip_sh) {
    using ST = typename Prec<T>::scale_t;
    using M = Mat4<T, C>;
    using Pr = Pairs<C>;
    if (nops == 0) return;
    if (sizeof(T) == 8) {
        for (int t = threadIdx.x; t < (I.SU + 1) * 4; t += kThreads) tip_sh[t] = m.tip[t];
        __syncthreads();
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p0 = p_first + wave * Pr::kPatterns;   // of the wavefront
    const int q = Pr::pattern(lane);
    const bool no_invar = I.invar[p0 + q] == 0.0;
    const typename M::A inv = M::load_same(m.inv_evec, lane);
    // the wavefront's part of a slot: its values and counters, and this lane's places in them
    constexpr uint32_t nv = 256 * sizeof(T);
    const uint32_t nc = (I.safe ? 64 : Pr::kPatterns) * sizeof(ST);
    const uint64_t vbase = (uint64_t)I.partial + (uint64_t)(p0 / Pr::kPatterns) * nv;
    const uint64_t cbase = (uint64_t)I.scale + (uint64_t)(p0 / Pr::kPatterns) * nc;
    auto part = [](uint64_t base, uint32_t slot, uint32_t bytes) { return buffer_of(base + ((uint64_t)slot << 8), bytes); };
    const uint32_t vat = lane * 16, sat = (I.safe ? q * C + Pr::cat(lane) : q) * sizeof(ST);
    const bool counting = I.safe || Pr::cat(lane) == 0;   // normal mode: a counter a pattern

    struct Kids {
        T v[2][4];                       // a slot's values
        T row[2][M::kRow];               // float: a tip's row of its lookup
        typename M::A e[2];              // the children's matrices
        int sc[2];                       // the pair's counters
    };
    struct States {
        unsigned w[2][M::kStates];
    };
    struct Desc {
        tile_u4 end;                     // dst, dsc, kind, root of the step itself
        tile_u4 tips, kids, kids_end;    // the step after next's
    };
    // float storage looks up a tip's row two steps ahead: its states come four ahead
    constexpr bool kTipsAhead = M::kRow > 1;
    const uint64_t tp = (uint64_t)tops;
    auto desc = [&](int o) {
        const uint64_t at = tp + (uint64_t)o * sizeof(TileOp);
        return Desc{load_u4(at + 32), load_u4(at + 128), load_u4(at + 144), load_u4(at + 160)};
    };
    auto load_states = [&](const tile_u4 tips, unsigned kind, States& st) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint64_t row = ((uint64_t)tips[2 * k + 1] << 32 | tips[2 * k]) + p0;
            if constexpr (M::kWords) {
                // of another child: taxon 0's, not used
                const auto* w = (const __attribute__((address_space(4))) unsigned*)row;
#pragma unroll
                for (int i = 0; i < M::kStates; i++) st.w[k][i] = w[i];
            } else if ((kind >> 2 * k & 3) == CHILD_TIP) {
                st.w[k][0] = ((const Hbm<uint8_t>*)row)[q];
            }
        }
    };
    const Hbm<T>* tab = (const Hbm<T>*)tables_g;
    auto load_tables = [&](unsigned kind, const States& st, Kids& in) {
        M::load(tab, table_size, lane, in.e);
#pragma unroll
        for (int k = 0; k < 2; k++)
            M::load_row(tab + k * table_size, (kind >> 2 * k & 3) == CHILD_TIP, st.w[k][0], lane, in.row[k]);
        tab += 2 * table_size;
    };
    // zeros (buffers of no bytes) for a child that is no slot
    auto load_slot = [&](const tile_u4 kids, int k, Kids& in) {
        const bool slot = kids[k] != kNoSlot;
        M::load_slot(part(vbase, kids[k], slot ? nv : 0), vat, in.v[k]);
        const Buffer counts = part(cbase, kids[2 + k], slot ? nc : 0);
        if (sizeof(ST) == 2) in.sc[k] = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(counts, sat, 0, 0);
        else in.sc[k] = (int)__builtin_amdgcn_raw_buffer_load_b32(counts, sat, 0, 0);
    };

    // even and odd steps have their own registers, since a copy would wait for
    // the loads. Steps past the end repeat the last one's TileOp (kTileAhead),
    // and read the tables of two steps more
    Desc d_even, d_odd;
    Kids even, odd;
    States st_even, st_odd;                // of the step; float: of the step after next
    T dad_even[4] = {}, dad_odd[4] = {};   // the last two dads
    int sc_even = 0, sc_odd = 0;
    {
        const tile_u4 k0 = load_u4(tp + 16), k1 = load_u4(tp + sizeof(TileOp) + 16);
        const tile_u4 e0 = load_u4(tp + 32), e1 = load_u4(tp + sizeof(TileOp) + 32);
        load_states(load_u4(tp), e0[2], st_even);
        load_states(load_u4(tp + sizeof(TileOp)), e1[2], st_odd);
        // slots last and unconditionally: the loop's first waits must not be
        // shorter than its later ones, which have stores to look past
        load_tables(e0[2], st_even, even);
        load_tables(e1[2], st_odd, odd);
        for (int k = 0; k < 2; k++) load_slot(k0, k, even);
        for (int k = 0; k < 2; k++) load_slot(k1, k, odd);
        d_even = desc(0);
        d_odd = desc(1);
        if constexpr (kTipsAhead) {
            load_states(d_even.tips, CHILD_TIP | CHILD_TIP << 2, st_even);
            load_states(d_odd.tips, CHILD_TIP | CHILD_TIP << 2, st_odd);
            d_even.tips = load_u4(tp + 4 * sizeof(TileOp));
            d_odd.tips = load_u4(tp + 5 * sizeof(TileOp));
        }
    }
    auto step = [&](int o, Desc& d, Kids& in, States& st, T(&dad)[4], int& dad_sc, const T(&last)[4], int last_sc) {
        T f[2][4];
        int sc = 0;
        const unsigned kinds = d.end[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const unsigned kind = kinds >> 2 * k & 3;
            if (kind == CHILD_TIP) {
                M::tip(in.e[k], in.row[k], st.w[k], d.end[3] >> k & 1, tip_sh, I.SU, lane, f[k]);
            } else if (kind == CHILD_LAST) {
                M::mul(in.e[k], last, f[k]);
                sc += last_sc;
            } else if (kind == CHILD_LAST2) {
                M::mul(in.e[k], dad, f[k]);
                sc += dad_sc;
            } else {
                M::mul(in.e[k], in.v[k], f[k]);
                sc += in.sc[k];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) f[0][i] *= f[1][i];
        M::mul(inv, f[0], dad);
        // a pattern is rescaled when all its categories (safe mode: the pair)
        // are below the threshold; tip-tip steps never
        const unsigned long long small = M::small(dad);
        if (small && kinds != (CHILD_TIP | CHILD_TIP << 2)) {
            int l = lane;
            asm("" : "+v"(l));   // masks of the lane are made here, not kept through the list
            if (I.safe) sc += M::template rescale<true>(dad, (small >> l & 1) && no_invar, l);
            else sc += M::template rescale<false>(
                dad, (small >> (l & ~Pr::kBits) & Pr::kMask) == Pr::kMask && no_invar, l);
        }
        dad_sc = sc;
        // the step after next's loads, then this step's stores: a wait for the
        // loads is then not one for these stores (a child that is a slot was
        // stored two steps ago or earlier)
        load_tables(d.kids_end[2], st, in);
#pragma unroll
        for (int k = 0; k < 2; k++)
            if ((d.kids_end[2] >> 2 * k & 3) == CHILD_SLOT) load_slot(d.kids, k, in);
        load_states(d.tips, kTipsAhead ? CHILD_TIP | CHILD_TIP << 2 : d.kids_end[2], st);
        M::store_slot(part(vbase, d.end[0], nv), vat, dad);
        if (counting) {
            const Buffer counts = part(cbase, d.end[1], nc);
            if (sizeof(ST) == 2) __builtin_amdgcn_raw_buffer_store_b16((unsigned short)sc, counts, sat, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b32(sc, counts, sat, 0, 0);
        }
        d = desc(o + 2);
        if constexpr (kTipsAhead) d.tips = load_u4(tp + (uint64_t)(o + 6) * sizeof(TileOp));
    };
    int o = 0;
    for (; o + 1 < nops; o += 2) {
        step(o, d_even, even, st_even, dad_even, sc_even, dad_odd, sc_odd);
        step(o + 1, d_odd, odd, st_odd, dad_odd, sc_odd, dad_even, sc_even);
    }
    if (o < nops) step(o, d_even, even, st_even, dad_even, sc_even, dad_odd, sc_odd);
}

// Branch ends for (p, c): node partial nv, dad partial (or tip vector from
// tip_sh) dv, the summed scale counter and, in safe mode, the per-category
// adjustment relative to the least-scaled category.
template <typename T, int N, int C>
__device__ inline void load_branch(const InstDev& I, plk_end node, plk_end dad, const double* tip_sh,
                                   int p, int c, double* nv, double* dv, int& minsc,
                                   double& adjust) {
    using ST = typename Prec<T>::scale_t;
    const T* partial = reinterpret_cast<const T*>(I.partial);
    const ST* scale = reinterpret_cast<const ST*>(I.scale);
    const bool safe = I.safe != 0;
    const T* nsrc = partial + Part<T, N, C>::at(I, node.id, p, c);
#pragma unroll
    for (int i = 0; i < N; i++) nv[i] = (double)nsrc[Part<T, N, C>::x(p, i)];
    int sc = scale[Part<T, N, C>::count_at(I, node.id, p, c)];
    if (dad.is_tip) {
        if (tip_sh) {   // callers that use a val-weighted lookup pass nullptr
            const int s = I.states[(size_t)dad.id * I.Ppad + p];
            const double* tp = tip_sh + s * N;
#pragma unroll
            for (int i = 0; i < N; i++) dv[i] = tp[i];
        }
    } else {
        const T* dsrc = partial + Part<T, N, C>::at(I, dad.id, p, c);
#pragma unroll
        for (int i = 0; i < N; i++) dv[i] = (double)dsrc[Part<T, N, C>::x(p, i)];
        sc += scale[Part<T, N, C>::count_at(I, dad.id, p, c)];
    }
    minsc = sc;
    adjust = 1.0;
    if (safe) {
        minsc = group_min_int<C>(sc);
        adjust = Prec<T>::safe_adjust(sc - minsc);
    }
}

// theta = node * dad (tip dad: its eigen-basis tip vector) and buffer_scale
// (computeLikelihoodBufferSIMD, tree/phylokernelnew.h:2091-2230)
template <typename T, int N, int C>
__device__ inline void theta_apply(const InstDev& I, plk_end node, plk_end dad, const double* tip_sh,
                                   int p, int c) {
    double nv[N], dv[N], adjust;
    int minsc;
    load_branch<T, N, C>(I, node, dad, tip_sh, p, c, nv, dv, minsc, adjust);
    T* th = reinterpret_cast<T*>(I.theta) + (size_t)p * (N * C) + c * N;
#pragma unroll
    for (int i = 0; i < N; i++) th[i] = (T)(nv[i] * dv[i] * adjust);
    if (c == 0) I.buffer_scale[p] = (double)minsc * Prec<T>::log_unit;
}

// Fused post-order traversal over the op list followed, per mode, by the
// branch lnL (computeLikelihoodBranchSIMD 2753-3104) or the theta buffer of
// the branch (node, dad).
template <typename T, int N, int C>
__global__ void __launch_bounds__(kThreads, 4)
k_traverse(InstDev I, ModelDev m, const TileOp* __restrict__ tops, int nops,
           const T* __restrict__ tables, int table_size, int mode, plk_end node, plk_end dad,
           const double* __restrict__ root_tab, double* __restrict__ block_sums) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int PB = kThreads / C;
    constexpr int block = N * C;
    const int c = threadIdx.x % C;
    const int p = blockIdx.x * PB + threadIdx.x / C;
    const bool live = p < I.Ppad;                            // every thread: PB divides Ppad

    static_assert(N == 4, "20 and 61 states have their own traversal kernels");
    dna_ops<T, C>(I, m, tops, nops, tables, table_size, blockIdx.x * PB, reinterpret_cast<double*>(smem));

    if (mode == MODE_PARTIALS) return;

    // ---- root stage ---------------------------------------------------------
    // MODE_BRANCH: root_tab = val[c][i] then, for a tip dad, lut[s][c][i] = val * tip
    // MODE_THETA:  the eigen-basis tip vectors
    double* root_sh = reinterpret_cast<double*>(smem);
    __syncthreads();
    if (mode == MODE_BRANCH) {
        const int root_size = block + (dad.is_tip ? (I.SU + 1) * block : 0);
        for (int t = threadIdx.x; t < root_size; t += kThreads) root_sh[t] = root_tab[t];
    } else if (dad.is_tip) {
        for (int t = threadIdx.x; t < (I.SU + 1) * N; t += kThreads) root_sh[t] = m.tip[t];
    }
    __syncthreads();
    double contrib = 0.0;
    if (live) {
        if (mode == MODE_THETA) {
            theta_apply<T, N, C>(I, node, dad, root_sh, p, c);
        } else {
            double nv[N], dv[N], adjust;
            int minsc;
            // a tip dad reads the val-weighted lookup lut[s][c][i] below instead of dv
            load_branch<T, N, C>(I, node, dad, nullptr, p, c, nv, dv, minsc, adjust);
            double lhc;
            if (dad.is_tip) {
                const int s = I.states[(size_t)dad.id * I.Ppad + p];
                const double* lut = root_sh + block + (s * C + c) * N;
                lhc = lut[0] * nv[0];
#pragma unroll
                for (int i = 1; i < N; i++) lhc = fma(lut[i], nv[i], lhc);
            } else {
                const double* val = root_sh + c * N;
                lhc = val[0] * dv[0] * nv[0];
#pragma unroll
                for (int i = 1; i < N; i++) lhc = fma(val[i] * dv[i], nv[i], lhc);
            }
            const double lh0 = I.safe ? group_sum_sumvec<C>(lhc * adjust) : group_sum_ordered<C>(lhc);
            if (c == 0) {
                const double lh = fabs(lh0) + I.invar[p];
                const int pobs = I.P - I.nasc;
                if (p < pobs) {
                    const double lnp = log(lh) + (double)minsc * Prec<T>::log_unit;
                    I.ptn_lh[p] = lnp;
                    contrib = lnp * I.freq[p];
                } else if (p < I.P) {
                    I.asc[4 * (p - pobs)] = Prec<T>::asc_scale(lh, minsc);
                }
            }
        }
    }
    if (mode == MODE_BRANCH) {
        double v[1] = {contrib};
        block_sum<1>(v, reinterpret_cast<double*>(smem));
        if (threadIdx.x == 0) block_sums[blockIdx.x] = v[0];
    }
}

// Patterns p0 .. p0 + n - 1 of a slot in the order of the interface: values
// [n][C][N], counters [n][safe ? C : 1], either may be null. Both are pinned
// host memory, written once and in order: bound by the host link.
template <typename T, int N, int C>
__global__ void __launch_bounds__(kThreads)
k_read_slot(InstDev I, int slot, int p0, int n, T* __restrict__ values, int32_t* __restrict__ counts) {
    using L = Part<T, N, C>;
    const T* partial = reinterpret_cast<const T*>(I.partial);
    const typename Prec<T>::scale_t* scale = reinterpret_cast<const typename Prec<T>::scale_t*>(I.scale);
    const size_t first = (size_t)blockIdx.x * kThreads + threadIdx.x, stride = (size_t)gridDim.x * kThreads;
    if (values)
        for (size_t t = first; t < (size_t)n * (N * C); t += stride) {
            const int p = p0 + (int)(t / (N * C)), c = (int)(t / N % C), i = (int)(t % N);
            values[t] = partial[L::at(I, slot, p, c) + L::x(p, i)];
        }
    const int nc = I.safe ? C : 1;
    if (counts)
        for (size_t t = first; t < (size_t)n * nc; t += stride)
            counts[t] = (int32_t)scale[L::count_at(I, slot, p0 + (int)(t / nc), (int)(t % nc))];
}

// ---------------------------------------------------------------------------
// Derivatives and lnL on the theta buffer (computeLikelihoodDervSIMD
// 2312-2551, computeLikelihoodFromBufferSIMD 3270-3343). Per pattern:
// lh = |sum_{c,i} val0 theta| + invar, d1 = sum val1 theta, d2 = sum val2 theta;
// df += f d1/lh, ddf += f (d2/lh - (d1/lh)^2), lnL += f (log lh + scale).
// One workgroup's share (patterns tile*PB ..) of the theta-buffer sums;
// out[0..2] = df, ddf and lnL partial sums (thread 0). val: LDS [3][N*C].
template <typename T, int N, int C>
__device__ inline void buffer_block(const InstDev& I, const ModelDev& m, double length, int mode,
                                    int tile, double* val, double* red, double* out) {
    constexpr int PB = kThreads / C;
    constexpr int block = N * C;
    for (int t = threadIdx.x; t < N * C; t += kThreads) {
        const int cc = t / N, i = t % N;
        const double cof = m.eval[i] * m.rates[cc];
        const double v0 = exp(cof * length) * m.props[cc];
        const double v1 = cof * v0;
        val[t] = v0;
        val[N * C + t] = v1;
        val[2 * N * C + t] = cof * v1;
    }
    __syncthreads();
    // With an odd state count and an even block, the reference's derivative
    // dot product (dotProductTriple, tree/phylokernelnew.h:668-716, called
    // with N = block at 2489-2491) adds the last (category, state) term twice
    // to lh, d1 and d2; the derivatives reproduce that for identical Newton
    // steps, while the lnL returned beside them uses the plain sum.
    constexpr bool kTwiceLast = (N & 1) && !((N * C) & 1);
    const int c = threadIdx.x % C;
    const int p = tile * PB + threadIdx.x / C;
    double lh = 0.0, d1 = 0.0, d2 = 0.0, lhq = 0.0;
    if (p < I.Ppad) {
        const T* th = reinterpret_cast<const T*>(I.theta) + (size_t)p * block + c * N;
        const double* v0 = val + c * N;
        const double* v1 = val + N * C + c * N;
        const double* v2 = val + 2 * N * C + c * N;
        constexpr int kUnroll = N <= 20 ? N : 4;   // 61 states: bounded register use
#pragma unroll kUnroll
        for (int i = 0; i < N; i++) {
            const double t = (double)th[i];
            lh = fma(v0[i], t, lh);
            if (mode == BUF_DERV) {
                d1 = fma(v1[i], t, d1);
                d2 = fma(v2[i], t, d2);
            }
        }
        lhq = lh;
        if (kTwiceLast && mode == BUF_DERV && c == C - 1) {
            const double t = (double)th[N - 1];
            lhq = fma(v0[N - 1], t, lh);
            d1 = fma(v1[N - 1], t, d1);
            d2 = fma(v2[N - 1], t, d2);
        }
    }
    lh = group_sum_ordered<C>(lh);
    if (mode == BUF_DERV) {
        d1 = group_sum_ordered<C>(d1);
        d2 = group_sum_ordered<C>(d2);
        lhq = kTwiceLast ? group_sum_ordered<C>(lhq) : lh;
    }
    double acc[3] = {0.0, 0.0, 0.0};
    const int pobs = I.P - I.nasc;
    if (c == 0 && p >= pobs && p < I.P) {
        // an unobserved constant pattern (+ASC): its probability and
        // derivatives, no weight of its own (tree/phylokernelnew.h:2497-2530, 3340-3358)
        const double bs = I.buffer_scale[p];
        double* a = I.asc + 4 * (p - pobs);
        a[0] = Prec<T>::asc_scale_log(fabs(lh) + I.invar[p], bs);
        if (mode == BUF_DERV) {
            a[1] = Prec<T>::asc_scale_log(fabs(lhq) + I.invar[p], bs);
            a[2] = Prec<T>::asc_scale_log(d1, bs);
            a[3] = Prec<T>::asc_scale_log(d2, bs);
        }
    }
    if (c == 0 && p < pobs) {
        lh = fabs(lh) + I.invar[p];
        const double f = I.freq[p];
        const double lnp = log(lh) + I.buffer_scale[p];
        if (mode == BUF_DERV) {
            const double inv = 1.0 / (kTwiceLast ? fabs(lhq) + I.invar[p] : lh);
            const double df_frac = d1 * inv, ddf_frac = d2 * inv;
            const double tmp1 = df_frac * f, tmp2 = ddf_frac * f;
            acc[0] = tmp1;
            acc[1] = tmp2 - tmp1 * df_frac;
            acc[2] = lnp * f;
        } else {
            I.ptn_lh[p] = lnp;
            acc[2] = lnp * f;
        }
    }
    block_sum<3>(acc, red);
    if (threadIdx.x == 0) {
        out[0] = acc[0];
        out[1] = acc[1];
        out[2] = acc[2];
    }
}

template <typename T, int N, int C>
__global__ void __launch_bounds__(kThreads)
k_buffer(InstDev I, ModelDev m, double length, int mode, double* __restrict__ block_sums) {
    __shared__ double val[3 * N * C];
    __shared__ double red[3 * (kThreads / 64)];
    buffer_block<T, N, C>(I, m, length, mode, blockIdx.x, val, red, block_sums + 3 * blockIdx.x);
}

// +ASC: pattern lnL of the observed patterns shifted by -log(1 - P(const)),
// the unobserved patterns' entries zeroed
__global__ void __launch_bounds__(kThreads)
k_asc_shift(double* __restrict__ ptn_lh, int pobs, int P, double corr) {
    const int p = blockIdx.x * kThreads + threadIdx.x;
    if (p < pobs) ptn_lh[p] -= corr;
    else if (p < P) ptn_lh[p] = 0.0;
}

// Fixed-order final reduction of per-workgroup partial sums: thread t adds
// entries t, t+256, ... in index order, then a fixed tree over threads.
__device__ inline void reduce_block(const double* __restrict__ in, int nblocks, int nvals,
                                    double* __restrict__ out, double* sh) {
    for (int j = 0; j < nvals; j++) {
        double s = 0.0;
        for (int b = threadIdx.x; b < nblocks; b += kThreads) s += in[(size_t)b * nvals + j];
        sh[threadIdx.x] = s;
        __syncthreads();
        for (int w = kThreads / 2; w >= 1; w >>= 1) {
            if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
            __syncthreads();
        }
        if (threadIdx.x == 0) out[j] = sh[0];
        __syncthreads();
    }
}

__global__ void __launch_bounds__(kThreads)
k_reduce(const double* __restrict__ in, int nblocks, int nvals, double* __restrict__ out) {
    __shared__ double sh[kThreads];
    reduce_block(in, nblocks, nvals, out, sh);
}

// RELL: out[b] = sum_p w[b][p] * ptn_lh[p], one workgroup per replicate.
__global__ void __launch_bounds__(kThreads)
k_rell(const float* __restrict__ w, const double* __restrict__ ptn_lh, int P, double* __restrict__ out) {
    __shared__ double sh[kThreads / 64];
    const float* wb = w + (size_t)blockIdx.x * P;
    double s = 0.0;
    for (int p = threadIdx.x; p < P; p += kThreads) s = fma((double)wb[p], ptn_lh[p], s);
    double v[1] = {s};
    block_sum<1>(v, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = v[0];
}

}  // namespace plkdev
