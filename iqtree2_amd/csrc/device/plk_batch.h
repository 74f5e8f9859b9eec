// Batched likelihood over many instances (partitions of a PhyloSuperTree,
// tree/phylosupertree.cpp:701-735, or independent requests) in one
// persistent launch.
//
// Work list: every (instance, pattern tile) pair with real patterns, ordered
// by the host largest-cost first (computePartitionOrder,
// tree/phylosupertree.cpp:654-690). Workgroups take the next tile from an
// atomic counter; a tile runs its instance's whole op list (transition tables
// of all ops of all instances were built by one k_prep_batch launch) and the
// root lnL of its instance's branch, and stores its lnL sum in its own slot.
// k_batch_reduce then adds each instance's tile sums in tile order, so the
// result does not depend on which workgroup ran which tile.
#pragma once
#include "plk_mfma.h"

namespace plkdev {

struct BatchItem {
    InstDev I;
    ModelDev m;
    const plk_op* ops;     // this instance's ops inside the batch op array
    const void* tables;    // [nops][2][table_size] storage precision (4 states: and two steps more)
    const TileOp* tops;    // the ops as dna_ops and prot_ops read them
    const double* root;    // val[C][n] then, for a tip dad, lut[SU+1][C][n]
    int nops;
    int table_size;
    int tile_begin;        // first global tile of this instance
    int ntiles;            // tiles with real patterns
    plk_end node, dad;
    int n, C, f32;
    int mode;              // BATCH_LNL: branch lnL; BATCH_THETA: theta buffer of the branch
};

enum { BATCH_LNL = 0, BATCH_THETA = 1 };

// Transition tables of a batch with k_prep_ops' arithmetic, and the root
// tables of k_prep_root. Workgroup (item, row) builds the tables of ops row,
// row + rows, ... of its item with the item's eigenvectors and tip vectors
// staged in LDS once; row 0 also writes the item's root tables and workgroup
// (0, 0) clears the work-list counters. LDS: evec n*n | tip SU*n | ex 2*C*n.
template <typename T>
__device__ inline void prep_child_table(const BatchItem& it, const plk_child ch, int k, const double* ev_sh,
                                        const double* tp_sh, const double* ex, T* step) {
    const int n = it.n, C = it.C, SU = it.I.SU, nn = n * n;
    T* out = step + (size_t)k * it.table_size;
    if (n == 4 && sizeof(T) == 8) {
        for (int t = threadIdx.x; t < C * nn; t += kThreads) {
            const int c = t / nn, r = t - c * nn;
            const T v = (T)(ev_sh[r] * ex[c * n + r % n]);
            dna_frag(C, c, r / n, r % n, k, [&](int at) { step[at] = v; });
        }
        return;
    }
    const bool prot = n == kProtN && sizeof(T) == 8;
    if (prot && (!ch.is_tip || !prot_lut(SU))) {
        for (int t = threadIdx.x; t < C * kProtBlocks; t += kThreads) {
            const int c = t / kProtBlocks, r = t - c * kProtBlocks;
            int x, i;
            prot_block_index(r, x, i);
            step[(2 * c + k) * kProtKid + r] = x < 0 ? (T)0 : (T)(ev_sh[x * n + i] * ex[c * n + i]);
        }
        return;
    }
    if (!ch.is_tip) {
        if (n == kProtN) {
            // the matrix-core tile's fragment order
            for (int t = threadIdx.x; t < C * kProtFrag; t += kThreads) {
                const int c = t / kProtFrag;
                int x, i;
                prot_frag_index(t - c * kProtFrag, x, i);
                out[t] = x < 0 ? (T)0 : (T)(ev_sh[x * n + i] * ex[c * n + i]);
            }
            return;
        }
        for (int t = threadIdx.x; t < C * nn; t += kThreads) {
            const int c = t / nn, r = t - c * nn, x = r / n, i = r - x * n;
            out[t] = (T)(ev_sh[x * n + i] * ex[c * n + i]);
        }
        return;
    }
    const int nv = C * n;
    for (int t = threadIdx.x; t < (SU + 1) * nv; t += kThreads) {
        const int s = t / nv, c = (t / n) % C, x = t % n;
        double v;
        if (s == SU) {
            v = 1.0;
        } else {
            const double* ev = ev_sh + x * n;
            const double* e = ex + c * n;
            const double* tp = tp_sh + s * n;
            v = ev[0] * e[0] * tp[0];
            for (int i = 1; i < n; i++) v += ev[i] * e[i] * tp[i];
        }
        if (prot) step[(2 * c + k) * kProtKid + s * n + x] = (T)v;
        else out[t] = (T)v;
    }
}

__global__ void __launch_bounds__(kThreads)
k_prep_batch(const BatchItem* __restrict__ items, const double* __restrict__ lengths,
             double* __restrict__ roots, unsigned* __restrict__ counters, int ncounters) {
    extern __shared__ double sh[];
    if (blockIdx.x == 0 && blockIdx.y == 0)
        for (int t = threadIdx.x; t < ncounters; t += kThreads) counters[t] = 0u;
    const int i = blockIdx.x;
    const BatchItem& it = items[i];
    const int n = it.n, C = it.C, SU = it.I.SU, nn = n * n, nv = C * n;
    double* ev_sh = sh;
    double* tp_sh = ev_sh + nn;
    double* ex = tp_sh + SU * n;
    if ((int)blockIdx.y < it.nops) {
        for (int t = threadIdx.x; t < nn; t += kThreads) ev_sh[t] = it.m.evec[t];
        for (int t = threadIdx.x; t < SU * n; t += kThreads) tp_sh[t] = it.m.tip[t];
    }
    for (int o = blockIdx.y; o < it.nops; o += gridDim.y) {
        const plk_op op = it.ops[o];
        __syncthreads();   // staging visible, the previous op's ex consumed
        for (int t = threadIdx.x; t < 2 * nv; t += kThreads) {
            const int k = t / nv, c = (t / n) % C, q = t % n;
            ex[t] = exp(it.m.eval[q] * (it.m.rates[c] * op.child[k].length));
        }
        __syncthreads();
        for (int k = 0; k < 2; k++) {
            const size_t off = (size_t)2 * o * it.table_size;
            void* tables = hbm(const_cast<void*>(it.tables));
            if (it.f32)
                prep_child_table<float>(it, op.child[k], k, ev_sh, tp_sh, ex + k * nv, reinterpret_cast<float*>(tables) + off);
            else
                prep_child_table<double>(it, op.child[k], k, ev_sh, tp_sh, ex + k * nv, reinterpret_cast<double*>(tables) + off);
        }
        if ((n == 4 || (n == kProtN && !it.f32)) && threadIdx.x == 0) {
            TileOp* tops = hbm(const_cast<TileOp*>(it.tops));
            make_tile_op(it.I, it.ops, o, it.nops, tops);
        }
    }
    if (blockIdx.y != 0) return;
    double* out = const_cast<double*>(it.root);
    const double len = lengths[i];
    for (int t = threadIdx.x; t < nv; t += blockDim.x) {
        const int c = t / n, q = t % n;
        out[t] = exp(it.m.eval[q] * (it.m.rates[c] * len)) * it.m.props[c];
    }
    if (!it.dad.is_tip) return;
    for (int t = threadIdx.x; t < (SU + 1) * nv; t += blockDim.x) {
        const int q = t % n, c = (t / n) % C, s = t / nv;
        out[nv + t] = exp(it.m.eval[q] * (it.m.rates[c] * len)) * it.m.props[c] * it.m.tip[s * n + q];
    }
}

// Branch ends streamed one state at a time (20 states keep no per-thread
// state arrays), with the arithmetic of load_branch + the root / theta code
// of k_traverse and k_root_stream. MODE_BRANCH returns the pattern's
// category sum (every lane) and the scale minimum; MODE_THETA writes theta
// and buffer_scale (tip dads read tip_eig).
template <typename T, int N, int C>
__device__ inline double branch_end_stream(const InstDev& I, plk_end node, plk_end dad, int mode,
                                           const double* root_sh, int p, int c,
                                           const double* __restrict__ tip_eig, int* minsc_out = nullptr) {
    using ST = typename Prec<T>::scale_t;
    constexpr int block = N * C;
    const T* partial = reinterpret_cast<const T*>(I.partial);
    const ST* scale = reinterpret_cast<const ST*>(I.scale);
    const bool safe = I.safe != 0;
    const size_t sidx = safe ? (size_t)p * C + c : (size_t)p;
    using L = Part<T, N, C>;
    const T* nv = partial + L::at(I, node.id, p, c);
    int sc = scale[(size_t)node.id * I.scale_stride + sidx];
    const T* dv = nullptr;
    int s = 0;
    if (dad.is_tip) {
        s = I.states[(size_t)dad.id * I.Ppad + p];
    } else {
        dv = partial + L::at(I, dad.id, p, c);
        sc += scale[(size_t)dad.id * I.scale_stride + sidx];
    }
    int minsc = sc;
    double adjust = 1.0;
    if (safe) {
        minsc = group_min_int<C>(sc);
        adjust = Prec<T>::safe_adjust(sc - minsc);
    }
    if (mode == MODE_THETA) {
        T* th = reinterpret_cast<T*>(I.theta) + (size_t)p * block + c * N;
        if (dad.is_tip) {
            const double* tp = tip_eig + s * N;
#pragma unroll 4
            for (int i = 0; i < N; i++) th[i] = (T)((double)nv[L::x(p, i)] * tp[i] * adjust);
        } else {
#pragma unroll 4
            for (int i = 0; i < N; i++) th[i] = (T)((double)nv[L::x(p, i)] * (double)dv[L::x(p, i)] * adjust);
        }
        if (c == 0) I.buffer_scale[p] = (double)minsc * Prec<T>::log_unit;
        return 0.0;
    }
    double lhc;
    if (dad.is_tip) {
        const double* lut = root_sh + block + (s * C + c) * N;
        lhc = lut[0] * (double)nv[0];
#pragma unroll 1
        for (int i = 1; i < N; i++) lhc = fma(lut[i], (double)nv[L::x(p, i)], lhc);
    } else {
        const double* val = root_sh + c * N;
        lhc = val[0] * (double)dv[0] * (double)nv[0];
#pragma unroll 1
        for (int i = 1; i < N; i++) lhc = fma(val[i] * (double)dv[L::x(p, i)], (double)nv[L::x(p, i)], lhc);
    }
    if (minsc_out) *minsc_out = minsc;
    return safe ? group_sum_sumvec<C>(lhc * adjust) : group_sum_ordered<C>(lhc);
}

// 16-pattern MFMA sub-tiles of a protein batch tile
constexpr int kBatchSub = 4;

// Dynamic LDS bytes batch_tile uses for one item shape: what its op list needs
// (4 states: dna_ops; 20 states: prot_ops, or in float storage the maxima of
// prot_ops_tile, 2 x kBatchSub x C x 16), then the root tables.
__host__ __device__ inline size_t batch_smem_bytes(int n, int C, int SU, int table_size, size_t elem) {
    const size_t root = (size_t)(SU + 2) * n * C * 8;
    if (n == kCodonN) return (size_t)2 * n * kCodonStride * elem;   // E | U^-1; root rows stay in HBM
    if (n == kProtN && elem == 8) {
        const size_t ops = prot_ops_smem(SU, 4);
        return ops > root ? ops : root;
    }
    if (n == kProtN) {
        const size_t mf = (size_t)2 * kBatchSub * C * 16 * elem;
        return mf > root ? mf : root;
    }
    const size_t ops = dna_ops_smem(SU);
    return ops > root ? ops : root;
}

// patterns per work-list tile: one per C threads (four 16-pattern protein
// matrix-core tiles, one codon tile)
__host__ __device__ constexpr int batch_tile_patterns(int C) { return kThreads / C; }

// all ops of one tile of one item, then its root lnL; returns the tile's
// lnL sum (thread 0)
template <typename T, int N, int C>
__device__ __forceinline__ double batch_tile(const BatchItem& it, int tile, unsigned char* smem) {
    constexpr int PB = batch_tile_patterns(C);
    constexpr int block = N * C;
    const InstDev I = on_hbm(it.I);
    const ModelDev m = on_hbm(it.m);
    const int c = threadIdx.x % C;
    const int p = tile * PB + (int)threadIdx.x / C;
    const T* tables = hbm(reinterpret_cast<const T*>(it.tables));
    const plk_op* ops = hbm(it.ops);
    __syncthreads();
    if constexpr (N == kCodonN) {
        // codon: the lone kernel's matrix-core tile, one pass per rate
        // category (each category's scaling is its own)
        constexpr int S = kCodonStride;
        static_assert(PB == kCodonTile, "batch tile must be one codon tile");
        T* e_m = reinterpret_cast<T*>(smem);
        T* inv_m = e_m + N * S;
        stage_lds<N * N>(inv_m, m.inv_evec, N * N, [](int t) { return (t / N) * S + t % N; });
        __syncthreads();
        for (int cc = 0; cc < C; cc++)
            codon_ops_tile<T>(I, ops, it.nops, tables, it.table_size, cc, tile * PB, e_m, inv_m);
    } else if constexpr (N == 20 && sizeof(T) == 8) {
        // a workgroup's 32 patterns twice
        static_assert(PB == 2 * kProtPatterns, "two blocks a tile");
        for (int h = 0; h < 2; h++)
            prot_ops<C>(I, m, it.tops, it.nops, tables, it.table_size, tile * PB + h * kProtPatterns, smem);
    } else if constexpr (N == 20) {
        // protein: the matrix-core tile of the lone traversal kernel, every
        // wave one category of four 16-pattern sub-tiles
        static_assert(PB == kBatchSub * kMfmaTile, "batch tile must be kBatchSub MFMA tiles");
        prot_ops_tile<T, C, kBatchSub>(I, m.inv_evec, ops, it.nops, tables, it.table_size,
                                       reinterpret_cast<T*>(smem), tile * PB);
    } else {
        dna_ops<T, C>(I, m, it.tops, it.nops, tables, it.table_size, tile * PB, reinterpret_cast<double*>(smem));
    }
    double* root_sh = reinterpret_cast<double*>(smem);
    const plk_end node = it.node, dad = it.dad;
    __syncthreads();
    if (it.mode == BATCH_THETA) {
        // computeLikelihoodBufferSIMD's theta: tip dads read the tip vectors
        // (the streamed form reads them from HBM)
        if constexpr (N == 4) {
            if (dad.is_tip)
                for (int t = threadIdx.x; t < (I.SU + 1) * N; t += kThreads) root_sh[t] = m.tip[t];
            __syncthreads();
            theta_apply<T, N, C>(I, node, dad, root_sh, p, c);
        } else {
            branch_end_stream<T, N, C>(I, node, dad, MODE_THETA, root_sh, p, c, m.tip);
        }
        return 0.0;
    }
    if constexpr (N == kCodonN) {
        // 61-state lookup rows (121 KB for a tip dad) stay in HBM, as k_root_stream reads them
        root_sh = hbm(const_cast<double*>(it.root));
    } else {
        const int root_size = block + (dad.is_tip ? (I.SU + 1) * block : 0);
        for (int t = threadIdx.x; t < root_size; t += kThreads) root_sh[t] = hbm(it.root)[t];
        __syncthreads();
    }
    double contrib = 0.0;
    double lh0;
    int minsc;
    if constexpr (N != 4) {
        // streamed (no per-thread state arrays), same arithmetic as below
        lh0 = branch_end_stream<T, N, C>(I, node, dad, MODE_BRANCH, root_sh, p, c, m.tip, &minsc);
    } else {
        double nv[N], dv[N], adjust;
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
        lh0 = I.safe ? group_sum_sumvec<C>(lhc * adjust) : group_sum_ordered<C>(lhc);
    }
    if (c == 0) {
        const double lh = fabs(lh0) + I.invar[p];
        const double lnp = log(lh) + (double)minsc * Prec<T>::log_unit;
        if (p < I.P) {
            I.ptn_lh[p] = lnp;
            contrib = lnp * I.freq[p];
        }
    }
    double v[1] = {contrib};
    block_sum<1>(v, reinterpret_cast<double*>(smem));
    return v[0];
}

// Instance classes a batch kernel is built for (bit mask). BC_ALL is the
// fused DNA + protein launch; codon tiles (63 KB of LDS) always run in a
// launch of their own class, so they do not lower the others' occupancy.
enum BatchClass {
    BC_DNA64 = 1, BC_PROT64 = 2, BC_DNA32 = 4, BC_PROT32 = 8, BC_ALL = 15, BC_F64 = 3, BC_F32 = 12,
    BC_COD64 = 16, BC_COD32 = 32
};
constexpr int kBatchClasses = 6;

__host__ __device__ inline int batch_class(int n, int f32) {
    if (n == 4) return f32 ? BC_DNA32 : BC_DNA64;
    if (n == 20) return f32 ? BC_PROT32 : BC_PROT64;
    return f32 ? BC_COD32 : BC_COD64;
}

// The tile list of one launch in kXcds segments, one per XCD of the device:
// the host places all of an item's tiles in one segment (its transition
// tables then sit in one XCD's L2 instead of every XCD fetching them),
// items bin-packed by cost. Segment q holds tiles [b[q], b[q + 1]).
constexpr int kXcds = 8;
struct XcdSplit {
    int b[kXcds + 1];
};

// Persistent workgroups over the tiles of `xs`. A workgroup takes tiles from
// its own XCD's segment (workgroups are dispatched to the XCDs round-robin,
// so blockIdx.x % kXcds), then from the others' in turn until every segment
// is drained; every workgroup ends after trying each segment's counter. MASK
// names the instance classes the launch may meet; a tile's code path is
// uniform across its workgroup.
// The classes with protein in FP64 are held to 3 waves per SIMD (168
// registers), the others of DNA and protein to 4, without spills in their
// loops; the compiler's own choice left each one wave or more lower. Classes
// of one storage have a fused kernel of their own (the tiles of 500 partitions:
// FP64 2,940 us fused, 975 + 2,040 in two launches, FP32 2,880 and 645 + 2,130).
template <int MASK>
__global__ void __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(MASK & ~BC_ALL ? 1 : MASK & BC_PROT64 ? 3 : 4)))
k_batch(const BatchItem* __restrict__ items, const int* __restrict__ tile_item, XcdSplit xs,
        unsigned* __restrict__ counters, double* __restrict__ tile_sums) {
    extern __shared__ __align__(16) unsigned char smem[];
    // thread 0's scheduling state lives in LDS, so no register stays live
    // across the tiles
    __shared__ int next_sh, tried_sh, bound_sh[kXcds + 1];
    if (threadIdx.x <= kXcds) bound_sh[threadIdx.x] = xs.b[threadIdx.x];
    if (threadIdx.x == 0) tried_sh = 0;   // segments found empty
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) {
            const int home = blockIdx.x % kXcds;
            int g = -1, tried = tried_sh;
            while (tried < kXcds) {
                const int q = (home + tried) % kXcds;
                const int t = bound_sh[q] + (int)atomicAdd(&counters[q], 1u);
                if (t < bound_sh[q + 1]) {
                    g = t;
                    break;
                }
                tried++;
            }
            tried_sh = tried;
            next_sh = g;
        }
        __syncthreads();
        // wave-uniform by construction; readfirstlane lets the item's fields
        // live in scalar registers
        const int g = __builtin_amdgcn_readfirstlane(next_sh);
        if (g < 0) break;
        const int i = __builtin_amdgcn_readfirstlane(tile_item[g]);
        const BatchItem& it = items[i];
        const int tile = g - it.tile_begin;
        const int cls = batch_class(it.n, it.f32);
        double s = 0.0;
        if ((MASK & BC_DNA64) && cls == BC_DNA64) s = batch_tile<double, 4, 4>(it, tile, smem);
        else if ((MASK & BC_PROT64) && cls == BC_PROT64) s = batch_tile<double, 20, 4>(it, tile, smem);
        else if ((MASK & BC_DNA32) && cls == BC_DNA32) s = batch_tile<float, 4, 4>(it, tile, smem);
        else if ((MASK & BC_PROT32) && cls == BC_PROT32) s = batch_tile<float, 20, 4>(it, tile, smem);
        else if ((MASK & BC_COD64) && cls == BC_COD64) s = batch_tile<double, kCodonN, 4>(it, tile, smem);
        else if ((MASK & BC_COD32) && cls == BC_COD32) s = batch_tile<float, kCodonN, 4>(it, tile, smem);
        if (threadIdx.x == 0) tile_sums[g] = s;
    }
}

// lnl[i] = sum of item i's tile sums in tile order (one thread per item)
__global__ void __launch_bounds__(kThreads)
k_batch_reduce(const BatchItem* __restrict__ items, int nitems, const double* __restrict__ tile_sums,
               double* __restrict__ lnl) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nitems) return;
    double s = 0.0;
    for (int t = 0; t < items[i].ntiles; t++) s += tile_sums[items[i].tile_begin + t];
    lnl[i] = s;
}

// ---------------------------------------------------------------------------
// Batched theta-buffer evaluations: one item = (instance, branch length), the
// derivative and lnL sums of computeLikelihoodDervSIMD for each. Every item
// is split into the same pattern tiles as a lone plk_likelihood_derv launch
// and its tile sums are reduced with the same fixed-order tree, so an item's
// result is bit-identical to the single-instance call whatever else shares
// the batch. One launch per (precision, states, categories) shape present.
struct DervItem {
    InstDev I;
    ModelDev m;
    double length;
    int tile_begin;   // first global tile
    int ntiles;       // Ppad / (kThreads / C)
};

template <typename T, int N, int C>
__global__ void __launch_bounds__(kThreads)
k_derv_batch(const DervItem* __restrict__ items, const int* __restrict__ tile_item, int tile_begin,
             double* __restrict__ tile_sums) {
    __shared__ double val[3 * N * C];
    __shared__ double red[3 * (kThreads / 64)];
    const int g = tile_begin + blockIdx.x;
    const DervItem& it = items[tile_item[g]];
    buffer_block<T, N, C>(on_hbm(it.I), on_hbm(it.m), it.length, BUF_DERV, g - it.tile_begin, val, red,
                          tile_sums + 3 * (size_t)g);
}

// out[3i..3i+2] = df, ddf, lnL of item i (one workgroup per item)
__global__ void __launch_bounds__(kThreads)
k_derv_reduce(const DervItem* __restrict__ items, const double* __restrict__ tile_sums,
              double* __restrict__ out) {
    __shared__ double sh[kThreads];
    const DervItem& it = items[blockIdx.x];
    reduce_block(tile_sums + 3 * (size_t)it.tile_begin, it.ntiles, 3, out + 3 * (size_t)blockIdx.x, sh);
}

}  // namespace plkdev
