// tree.hip — short-range tree correction: Morton sort, linear octree, node moments, target
// groups and the wavefront-cooperative walk with the tabulated split force law.
//
// Reference semantics (paths relative to the reference tree):
//   driver       Cosmos/treecorrection.c:225-475 (chaining mesh of width >= cutoff, 27 neighbours)
//   tree         OST/ost.ver2.c:36-196 (monopole + quadrupole about the COM, rmax = max |x - COM|)
//   opening      OST/ost.ver2.c:296-306 (open when d^2 < rmax^2 / theta^2)
//   node force   OST/ost.ver2.c:247-277 (AddNode, with the y/z components of defect D1 restored)
//   pair force   OST/ost.ver2.c:279-293 (AddPar); both use the cutoff test d^2 <= rsphere^2
//   force law    OST/Model4TreeForce.c:34-46 (GetPointGrav / GetCellGrav, 4096-entry linear tables)
//
// MI355X design (not the reference's): one global octree per box instead of one tree per
// 4x4x4 cell. Particles are sorted by a 48-bit Morton key; the chaining cells are the
// octree nodes of level L (2^L per axis, width n/2^L >= cutoff). A node is the run of
// particles sharing a key prefix. All levels are built at once: the keys around a particle say which
// nodes begin at it, and the records stand level by level, the children of a node consecutive.
// Target groups are subtrees of <= 128 particles; one wavefront walks the 27 neighbouring
// cell trees for its group with a group-conservative opening test, stages accepted nodes
// and opened leaves in LDS, and evaluates the interactions lane-per-target.
#include "lagpm_internal.h"
#include "wave_ops.h"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

namespace {
using namespace lagpm_wave;

#ifndef WALK_THREADS_PER_CU
#define WALK_THREADS_PER_CU 1024
#endif
constexpr int WALK_THREADS = WALK_THREADS_PER_CU;  // one workgroup per CU (LDS: shared table + 16 wave lists)
constexpr int WALK_WAVES = WALK_THREADS / 64;
#ifndef WALK_PP_TAKE
#define WALK_PP_TAKE 4
#endif
#ifndef WALK_LSTACK
#define WALK_LSTACK 256
#endif
constexpr int PP_TAKE = WALK_PP_TAKE;  // particles a lane appends per round
constexpr int PP_CAP = 64 * PP_TAKE + 64;  // one round + 63 left over
constexpr int PC_CAP = 128;
constexpr int STACK_MAX = 8192;  // per-wave walk stack entries
constexpr int WALK_XCDS = LAGPM_WALK_XCDS;
constexpr int LSTACK = WALK_LSTACK;  // the first LSTACK entries of a wave's stack live in LDS, the rest in global memory
constexpr int WALK_MAX_ITERS = 1 << 20;  // per-group bound on 64-node pop rounds
// rmax: a leaf and an inner node of up to RMAX_EXACT_MAX particles get the exact largest distance
// of their particles from the com (the reference's node size); larger nodes get the bound
// max(|com_child - com| + rmax_child), which only opens such nodes somewhat earlier.
#ifndef RMAX_EXACT_MAX
#define RMAX_EXACT_MAX 128
#endif
constexpr float RAN_F = (float)(6.0 / 4096.0);
constexpr int TAB_LDS = LAGPM_LOG_BINS > 4096 ? LAGPM_LOG_BINS : 4096;

// Table bin and offset of a pair at squared distance r2 (see law_tables): uniform r bins need
// the square root; log r^2 bins take the exponent and 8 mantissa bits of r2.
template <bool LOGT>
__device__ inline int table_bin(float r2, float& t, float lam) {
    if constexpr (LOGT) {
        // Each bin holds the line c + s * r2 (bin 0 runs from r2 = 0, so it serves every r2 below
        // its node); bins beyond the cutoff hold zeros, so far pairs and the far-away dummies of a
        // partial chunk add nothing without a compare. r2 above the table is clamped to its last bin.
        // lam r2 >= 0, so its bit pattern orders like the value: one unsigned clamp of the bits to
        // [bin 0's node, just below 64] (a v_med3_u32) replaces a float clamp and an integer max.
        constexpr uint32_t LO = (uint32_t)LAGPM_LOG_BASE << LAGPM_LOG_SHIFT;
        constexpr uint32_t HI = ((uint32_t)(LAGPM_LOG_BASE + LAGPM_LOG_BINS) << LAGPM_LOG_SHIFT) - 1u;
        const uint32_t b = min(max(__float_as_uint(lam * r2), LO), HI);
        t = r2;
        // The bin, bits 15..30 of b, as one bit-field extract: the table address is then one
        // shift-and-add from it. Written as (b >> 15) the compiler turns the shift and the
        // address's scaling by 8 into a shift, a mask and an add: one more operation per pair.
        static_assert(LAGPM_LOG_SHIFT == 15, "the extract below takes bits 15..30");
        uint32_t f;
        asm("v_bfe_u32 %0, %1, 15, 16" : "=v"(f) : "v"(b));
        return (int)f - (int)LAGPM_LOG_BASE;
    } else {
        const float r = __builtin_amdgcn_sqrtf(r2);
        const int nt = min((int)(r * (1.0f / RAN_F)), 4095);
        t = r - (float)nt * RAN_F;
        return nt;
    }
}
template <bool LOGT>
__device__ inline int table_bin64(double r2, double& t, float lam) {
    if constexpr (LOGT) {
        const double r2c = fmin((double)lam * r2, 63.99);
        t = r2;  // bins hold c + s * r2, zero beyond the cutoff (see table_bin)
        return max((int)(__float_as_uint((float)r2c) >> LAGPM_LOG_SHIFT) - (int)LAGPM_LOG_BASE, 0);
    } else {
        const double ran = 6.0 / 4096.0;
        const double r = sqrt(r2);
        const int nt = min((int)(r / ran), 4095);
        t = r - nt * ran;
        return nt;
    }
}

__device__ inline uint64_t spread3(uint32_t v) {
    uint64_t x = v & 0xffffu;
    x = (x | (x << 32)) & 0x1f00000000ffffull;
    x = (x | (x << 16)) & 0x1f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}
__device__ inline uint32_t compact3(uint64_t x) {
    x &= 0x1249249249249249ull;
    x = (x | (x >> 2)) & 0x10c30c30c30c30c3ull;
    x = (x | (x >> 4)) & 0x100f00f00f00f00full;
    x = (x | (x >> 8)) & 0x1f0000ff0000ffull;
    x = (x | (x >> 16)) & 0x1f00000000ffffull;
    x = (x | (x >> 32)) & 0x1fffffull;
    return (uint32_t)x;
}
__device__ inline uint32_t quant(double x, double s) {
    double q = floor(x * s);
    if (q < 0) q = 0;
    if (q > 65535.0) q = 65535.0;
    return (uint32_t)q;
}
__device__ inline int key_shift(int level) { return 3 * (LAGPM_KEY_BITS - level); }
// number of leading octal digits two keys share (16 when equal)
__device__ inline int common_digits(uint64_t a, uint64_t b) {
    uint64_t d = a ^ b;
    if (d == 0) return LAGPM_KEY_BITS;
    int p = 63 - __clzll(d);
    return (47 - p) / 3;
}
// first index in [lo, hi) whose prefix (key >> sh) exceeds pfx
__device__ inline size_t upper_bound_pfx(const uint64_t* __restrict__ K, size_t lo, size_t hi, uint64_t pfx, int sh) {
    while (lo < hi) {
        size_t mid = lo + ((hi - lo) >> 1);
        if ((K[mid] >> sh) > pfx) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}
// first index in [lo, hi) whose prefix is >= pfx
__device__ inline size_t lower_bound_pfx(const uint64_t* __restrict__ K, size_t lo, size_t hi, uint64_t pfx, int sh) {
    while (lo < hi) {
        size_t mid = lo + ((hi - lo) >> 1);
        if ((K[mid] >> sh) >= pfx) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

// Morton keys of the positions and the identity permutation. (The Hubble drag of the step's front,
// v *= drag[0], Cosmos/globalT.c:102-110, rides in the gather after the sort.)
__global__ void keys_kernel(const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
                            size_t np, double s, uint64_t* __restrict__ key, uint32_t* __restrict__ perm) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    key[i] = spread3(quant(x[i], s)) | (spread3(quant(y[i], s)) << 1) | (spread3(quant(z[i], s)) << 2);
    perm[i] = (uint32_t)i;
}

// all particle arrays into the new order in one pass (one permutation load, seven gathers in flight)
struct gather_set {
    const double* src[6];
    double* dst[6];
    const uint32_t* id;
    uint32_t* id_dst;
};
// The sources of neighbouring outputs share cache lines (the order changes little between steps),
// so the gather gives each XCD one contiguous range of outputs (lagpm_wave::xcd_block): the lines
// those outputs read are fetched into one L2 instead of into several. With drag, the velocities
// are multiplied by drag[0] on the way (the Hubble drag of the step's front), a pass over them
// that the keys would otherwise make.
__global__ void gather_all_kernel(gather_set g, const uint32_t* __restrict__ perm, size_t np,
                                  const double* __restrict__ drag) {
    const size_t i = (size_t)lagpm_wave::xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const uint32_t p = perm[i];
    double v[6];
#pragma unroll
    for (int a = 0; a < 6; a++) v[a] = g.src[a][p];
    const uint32_t id = g.id[p];
    if (drag) {
        const double f = drag[0];
        v[3] *= f;
        v[4] *= f;
        v[5] *= f;
    }
#pragma unroll
    for (int a = 0; a < 6; a++) g.dst[a][i] = v[a];
    g.id_dst[i] = id;
}

// The same gather in two halves, for a step front that runs them on two streams: the positions
// (which the deposit and the tree build wait for) and the velocities with the ids and the drag
// (which only the PM kick and the drift need, so they load beside the deposit and the build).
__global__ void gather_pos_kernel(gather_set g, const uint32_t* __restrict__ perm, size_t np) {
    const size_t i = (size_t)lagpm_wave::xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const uint32_t p = perm[i];
    double v[3];
#pragma unroll
    for (int a = 0; a < 3; a++) v[a] = g.src[a][p];
#pragma unroll
    for (int a = 0; a < 3; a++) g.dst[a][i] = v[a];
}
__global__ void gather_vel_kernel(gather_set g, const uint32_t* __restrict__ perm, size_t np,
                                  const double* __restrict__ drag) {
    const size_t i = (size_t)lagpm_wave::xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const uint32_t p = perm[i];
    double v[3];
#pragma unroll
    for (int a = 0; a < 3; a++) v[a] = g.src[3 + a][p];
    const uint32_t id = g.id[p];
    if (drag) {
        const double f = drag[0];
#pragma unroll
        for (int a = 0; a < 3; a++) v[a] *= f;
    }
#pragma unroll
    for (int a = 0; a < 3; a++) g.dst[3 + a][i] = v[a];
    g.id_dst[i] = id;
}

__device__ inline void tree_reset(int t, uint32_t* __restrict__ dsz, unsigned long long* __restrict__ counters) {
    if (t == DSZ_NODES || t == DSZ_GROUPS || t == DSZ_OVERFLOW || t == DSZ_DEEPER || t == DSZ_WALKOVF || t == DSZ_TICKET) dsz[t] = 0u;
    if (t >= DSZ_LVL && t < DSZ_LOFF) dsz[t] = 0u;
    if (t < 4) counters[t] = 0ull;
}

// node count on the device, clamped to the array capacity
__device__ inline size_t dev_count(const uint32_t* __restrict__ dsz, int which, size_t cap) {
    size_t c = dsz[which];
    return c < cap ? c : cap;
}

// ---------------------------------------------------------------------------------------
// Build from the sorted keys, all levels at once. Cells of the chaining level L are the roots; a
// node of more than nleaf particles above the depth limit D splits into its non-empty octants. Which
// nodes begin at particle f follows from the keys around it, whatever the other levels hold:
//   - the first level at which f starts a prefix of its own is l1 = max(L, 1 + digits shared with
//     f - 1); a node begins there if l1 = L, or if its parent, the prefix of l1 - 1 digits around f,
//     holds more than nleaf particles (as many of its neighbours within nleaf places either way say);
//   - below a node that begins at f, the next level's node begins at f too while f and f + nleaf share
//     the level's digits (the node then holds more than nleaf).
// So f's nodes are the levels l1 .. lk, and one pass over the particles counts them, a scan of the
// counts per block of TB_PART particles places them, and a second pass writes them: three launches
// where splitting level by level took two a level and a scan over the particles. Sort excluded, a
// build with its moments and groups took 0.38 ms for 128^3 clustered particles, 0.20 for 32^3; now
// 0.22 and 0.14.
// Records are level by level and in particle order within a level, so the children of a node are
// consecutive records; a node's own count (if it is no leaf) and number of children are filled in by
// the moments, which visit them anyway. The order is the same from run to run.
constexpr int TB_THREADS = 256;
constexpr int TB_ITEMS = 4;
constexpr int TB_PART = TB_THREADS * TB_ITEMS;  // particles per block
constexpr int TB_LEAF_MAX = 256;                // largest nleaf (lagpm_box_set_tuning)
constexpr int TB_ROWS = LAGPM_KEY_BITS + 3;     // counts per block: a row a level, all nodes, nodes beyond the limit
constexpr int TB_SEQ = TB_PART / 64;            // runs of 64 particles of a block, in particle order

// the block's keys with nleaf neighbours either way: s[i] is the key of particle base - nleaf + i
__device__ inline void tb_load_keys(const uint64_t* __restrict__ K, size_t N, long long base, int nleaf, uint64_t* s) {
    for (int i = threadIdx.x; i < TB_PART + 2 * nleaf; i += TB_THREADS) {
        const long long q = base - nleaf + i;
        s[i] = q >= 0 && q < (long long)N ? K[q] : 0ull;
    }
    __syncthreads();
}
// Levels l1 .. lk of the nodes that begin at particle f = base + i - nleaf (k = s + i, its key); lk <
// l1: none. cf: digits that f shares with f + nleaf (-1 past the end).
__device__ inline void tb_levels(const uint64_t* k, size_t f, size_t N, int nleaf, int L, int D, int& l1, int& lk, int& cf) {
    const int b = f == 0 ? -1 : common_digits(k[-1], k[0]);
    l1 = max(L, b + 1);
    lk = l1 - 1;
    cf = f + nleaf < N ? common_digits(k[0], k[nleaf]) : -1;
    if (l1 > D) return;
    if (l1 > L) {  // the parent (level b) holds f and f - 1: more than nleaf particles?
        const int sh = key_shift(b);
        const uint64_t pfx = k[0] >> sh;
        int lo = f < (size_t)nleaf ? -(int)f : -nleaf, hi = -1;  // first place of the parent among the nleaf before f
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if ((k[mid] >> sh) == pfx) hi = mid;
            else lo = mid + 1;
        }
        int a = 0, e = N - 1 - f < (size_t)nleaf ? (int)(N - 1 - f) : nleaf;  // last one among the nleaf after f
        while (a < e) {
            const int mid = (a + e + 1) >> 1;
            if ((k[mid] >> sh) == pfx) a = mid;
            else e = mid - 1;
        }
        if (a - lo + 1 <= nleaf) return;
    }
    lk = min(max(l1, cf + 1), D);
}

// Pass 1: the block's nodes per level, their sum, and the nodes that should split beyond the limit;
// beside it the cell roots cleared and (FP32 tree, pp non-null) the pp copy of the positions in units
// of the particle mass.
// pp is the FP32 copy of the positions for the tree, scaled by sc (rounded once from the FP64
// product): with the log-r^2 force tables sc = sqrt(lam), so a pair's r^2 in these units is lam r^2,
// the table variable, and needs no multiply in the pair loop. Everything the FP32 tree derives
// from pp (centres, second moments, node sizes, group boxes) is in the same units.
__global__ void __launch_bounds__(TB_THREADS) tree_count_kernel(const uint64_t* __restrict__ K, size_t N, int nleaf, int L, int D,
                                                                const double* __restrict__ x, const double* __restrict__ y,
                                                                const double* __restrict__ z, double sc, float4* __restrict__ pp,
                                                                int* __restrict__ cellroot, size_t ncell,
                                                                uint32_t* __restrict__ cnt, uint32_t nblk) {
    __shared__ uint64_t s[TB_PART + 2 * TB_LEAF_MAX];
    __shared__ uint32_t rows[TB_ROWS];
    for (size_t c = (size_t)blockIdx.x * TB_THREADS + threadIdx.x; c < ncell; c += (size_t)gridDim.x * TB_THREADS) cellroot[c] = -1;
    if (blockIdx.x >= nblk) return;
    if (threadIdx.x < TB_ROWS) rows[threadIdx.x] = 0u;
    const long long base = (long long)blockIdx.x * TB_PART;
    tb_load_keys(K, N, base, nleaf, s);
    const int lane = threadIdx.x & 63, nlev = D - L + 1;
    uint32_t mine = 0u;  // lane j: row j's count over this wave's particles
#pragma unroll
    for (int q = 0; q < TB_ITEMS; q++) {
        const int i = q * TB_THREADS + (int)threadIdx.x;
        const size_t f = (size_t)base + i;
        int l1 = 1, lk = 0, cf = -1;
        if (f < N) {
            tb_levels(s + nleaf + i, f, N, nleaf, L, D, l1, lk, cf);
            if (pp) pp[f] = make_float4((float)(x[f] * sc), (float)(y[f] * sc), (float)(z[f] * sc), 1.0f);
        }
        uint32_t all = 0u;
        for (int j = 0; j < nlev; j++) {
            const uint32_t c = (uint32_t)__popcll(__ballot(l1 <= L + j && L + j <= lk));
            all += c;
            if (lane == j) mine += c;
        }
        if (lane == nlev) mine += all;
        const uint32_t deep = (uint32_t)__popcll(__ballot(lk == D && cf >= D && D < LAGPM_KEY_BITS && l1 <= lk));
        if (lane == nlev + 1) mine += deep;
    }
    if (lane < nlev + 2) atomicAdd(&rows[lane], mine);
    __syncthreads();
    if ((int)threadIdx.x < nlev + 2) cnt[(size_t)threadIdx.x * nblk + blockIdx.x] = rows[threadIdx.x];
}
// exclusive scan of one row of n counts by a workgroup of 256; the total is returned to all threads
__device__ inline uint32_t block_row_scan(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, uint32_t n) {
    __shared__ uint32_t wsum[4];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    uint32_t carry = 0u;
    for (uint32_t c0 = 0; c0 < n; c0 += 2048) {
        uint32_t v[8], t = 0u;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t i = c0 + 8 * tid + k;
            v[k] = i < n ? in[i] : 0u;
            t += v[k];
        }
        int wt;
        uint32_t run = (uint32_t)wave_excl_scan((int)t, lane, wt);
        if (lane == 0) wsum[wid] = (uint32_t)wt;
        __syncthreads();
        uint32_t sum = 0u;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            if (w < wid) run += wsum[w];
            sum += wsum[w];
        }
        run += carry;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t i = c0 + 8 * tid + k;
            if (i < n) out[i] = run;
            run += v[k];
        }
        carry += sum;
        __syncthreads();
    }
    return carry;
}
// One workgroup per row: its offsets per block, and what the rows' totals say (a level's nodes, all
// nodes, whether the limit was met). The row of all nodes clears the other sizes and the counters.
__global__ void __launch_bounds__(256) tree_rows_kernel(const uint32_t* __restrict__ cnt, uint32_t* __restrict__ off, uint32_t nblk,
                                                        int L, int D, uint32_t* __restrict__ dsz,
                                                        unsigned long long* __restrict__ counters) {
    const int row = (int)blockIdx.x, nlev = D - L + 1;
    const uint32_t total = block_row_scan(cnt + (size_t)row * nblk, off + (size_t)row * nblk, nblk);
    const int t = (int)threadIdx.x;
    if (row < nlev) {
        if (t == 0) dsz[DSZ_LVL + L + row] = total;
    } else if (row == nlev) {
        if (t == 0) dsz[DSZ_NODES] = total;
        if (t == DSZ_GROUPS || t == DSZ_WALKOVF || t == DSZ_TICKET) dsz[t] = 0u;
        if (t <= LAGPM_KEY_BITS && (t < L || t > D)) dsz[DSZ_LVL + t] = 0u;
        if (t < 4) counters[t] = 0ull;
    } else if (t == 0) {
        dsz[DSZ_DEEPER] = total ? 1u : 0u;
    }
}
// Pass 2: the records. link: first particle, count (leaves; the moments fill in the others), first
// child record (0: a leaf; record 0 is a root), children (filled in); lev: level, and bit 8 for the
// first child of its parent; rop: the record of each pre-order number (first particle, then level).
__global__ void __launch_bounds__(TB_THREADS) tree_emit_kernel(const uint64_t* __restrict__ K, size_t N, int nleaf, int L, int D,
                                                               const uint32_t* __restrict__ off, uint32_t nblk, size_t cap,
                                                               uint32_t* __restrict__ dsz, int4* __restrict__ link,
                                                               int* __restrict__ lev, uint32_t* __restrict__ rop,
                                                               int* __restrict__ cellroot, int mcell) {
    __shared__ uint64_t s[TB_PART + 2 * TB_LEAF_MAX];
    __shared__ uint32_t wcnt[TB_SEQ][TB_ROWS];  // per run of 64 particles: its nodes per level, then the first record of each
    const int nlev = D - L + 1, lane = (int)(threadIdx.x & 63), wid = (int)(threadIdx.x >> 6);
    const bool over = dsz[DSZ_NODES] > cap || dsz[DSZ_DEEPER];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        uint32_t o = 0u;
        for (int l = 0; l <= LAGPM_KEY_BITS; l++) {
            dsz[DSZ_LOFF + l] = o;
            o += dsz[DSZ_LVL + l];
        }
        dsz[DSZ_OVERFLOW] = over ? 1u : 0u;  // the walk and the drift skip this box until it is redone
    }
    if (over) return;
    const long long base = (long long)blockIdx.x * TB_PART;
    tb_load_keys(K, N, base, nleaf, s);
    int l1[TB_ITEMS], lk[TB_ITEMS], cf[TB_ITEMS];
#pragma unroll
    for (int q = 0; q < TB_ITEMS; q++) {
        const int i = q * TB_THREADS + (int)threadIdx.x;
        const size_t f = (size_t)base + i;
        l1[q] = 1; lk[q] = 0; cf[q] = -1;
        if (f < N) tb_levels(s + nleaf + i, f, N, nleaf, L, D, l1[q], lk[q], cf[q]);
        uint32_t mine = 0u, all = 0u;
        for (int j = 0; j < nlev; j++) {
            const uint32_t c = (uint32_t)__popcll(__ballot(l1[q] <= L + j && L + j <= lk[q]));
            all += c;
            if (lane == j) mine = c;
        }
        if (lane == nlev) mine = all;
        if (lane <= nlev) wcnt[q * (TB_THREADS / 64) + wid][lane] = mine;
    }
    __syncthreads();
    if ((int)threadIdx.x <= nlev) {
        const int j = (int)threadIdx.x;
        uint32_t run = off[(size_t)j * nblk + blockIdx.x];
        if (j < nlev)
            for (int l = L; l < L + j; l++) run += dsz[DSZ_LVL + l];
        for (int q = 0; q < TB_SEQ; q++) {
            const uint32_t c = wcnt[q][j];
            wcnt[q][j] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TB_ITEMS; q++) {
        const int i = q * TB_THREADS + (int)threadIdx.x, sq = q * (TB_THREADS / 64) + wid;
        const size_t f = (size_t)base + i;
        const uint64_t* k = s + nleaf + i;
        auto below = [](unsigned long long m) {  // lanes below this one in m
            return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
        };
        uint32_t pre = wcnt[sq][nlev];
        for (int j = 0; j < nlev; j++) pre += below(__ballot(l1[q] <= L + j && L + j <= lk[q]));
        uint32_t r = wcnt[sq][0] + below(__ballot(l1[q] <= L && L <= lk[q]));
        for (int j = 0; j < nlev; j++) {
            const int l = L + j;
            const bool act = l1[q] <= l && l <= lk[q];
            uint32_t rn = 0u;
            if (j + 1 < nlev) rn = wcnt[sq][j + 1] + below(__ballot(l1[q] <= l + 1 && l + 1 <= lk[q]));
            if (act) {
                uint32_t count = 0u;
                const bool leaf = l == lk[q];
                if (leaf) {
                    const int sh = key_shift(l);
                    const uint64_t pfx = k[0] >> sh;
                    if (cf[q] < l) {  // ends within nleaf places
                        int a = 0, e = N - 1 - f < (size_t)nleaf ? (int)(N - 1 - f) : nleaf;
                        while (a < e) {
                            const int mid = (a + e + 1) >> 1;
                            if ((k[mid] >> sh) == pfx) a = mid;
                            else e = mid - 1;
                        }
                        count = (uint32_t)(a + 1);
                    } else {  // more than nleaf particles in one finest cell
                        count = (uint32_t)(upper_bound_pfx(K, f + nleaf, N, pfx, sh) - f);
                    }
                }
                link[r] = make_int4((int)f, (int)count, leaf ? 0 : (int)rn, 0);
                lev[r] = l | (l > l1[q] ? 256 : 0);
                rop[pre + (uint32_t)(l - l1[q])] = r;
                if (l == L) {
                    const uint64_t cell = k[0] >> key_shift(L);
                    cellroot[compact3(cell) + (size_t)mcell * (compact3(cell >> 1) + (size_t)mcell * compact3(cell >> 2))] = (int)r;
                }
            }
            r = rn;
        }
    }
}
// A record's children: record fc and those after it up to the next first child (bit 8 of lev) or the
// level's end. Every lane of the record's row of 8 calls it (sub: its index in the row).
__device__ inline int row_children(const int* __restrict__ lev, int fc, int sub, uint32_t level_end) {
    const uint32_t c = (uint32_t)fc + (uint32_t)sub;
    const bool stop = fc == 0 || c >= level_end || (sub > 0 && (lev[c] & 256));
    const uint32_t row = (uint32_t)(__ballot(stop) >> (threadIdx.x & 56)) & 0xffu;
    return fc == 0 ? 0 : (row ? __ffs((int)row) - 1 : 8);
}

__device__ inline void kahan(float& s, float& c, float v) {
    float y = v - c;
    float t = s + y;
    c = (t - s) - y;
    s = t;
}

// FP32 moments, one level per launch (deepest first), 8 lanes per node: the lanes take
// the node's particles (or children) in turn, so a row's loads are consecutive particles, and the
// row's partial sums meet in a butterfly. Each lane sums with Kahan compensation, relative to the
// node's first member (or first child's com); the compensated lane sums are then added in a fixed
// order, so the moments are deterministic. Leaves read their particles; inner nodes read their
// children's moments, consecutive records which the previous level's launch wrote, and get their
// count and number of children on the way (and inner nodes of at most RMAX_EXACT_MAX particles read
// their particles again for the exact rmax).
constexpr int MOM_ROW = 8;  // lanes per node: a leaf's <= 32 particles are 4 per lane, an inner node's <= 8 children 1
__device__ inline float row_sum(float v) {
#pragma unroll
    for (int o = MOM_ROW / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, MOM_ROW);
    return v;
}
__device__ inline float row_max(float v) {
#pragma unroll
    for (int o = MOM_ROW / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, MOM_ROW));
    return v;
}
__device__ inline int row_sum(int v) {
#pragma unroll
    for (int o = MOM_ROW / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, MOM_ROW);
    return v;
}
// every lane of the record's row calls this with its index `sub` in the row
__device__ inline void moments_f32_node(size_t r8, int sub, uint32_t level_end, const float4* __restrict__ pp,
                                        const int* __restrict__ lev, int4* __restrict__ link, float4* __restrict__ geo,
                                        float4* __restrict__ q0, float4* __restrict__ q1) {
    int4 nd = link[r8];
    const int nch = row_children(lev, nd.z, sub, level_end);
    float M = 0, cM = 0, Sx = 0, cx = 0, Sy = 0, cy = 0, Sz = 0, cz = 0;
    float Q[6] = {0, 0, 0, 0, 0, 0}, cQ[6] = {0, 0, 0, 0, 0, 0};
    float r2max = 0.f, rbound = 0.f;
    float3 cm;
    if (nch == 0) {
        const float4 r = pp[nd.x];
        for (int p = nd.x + sub; p < nd.x + nd.y; p += MOM_ROW) {
            const float4 a = pp[p];
            kahan(M, cM, a.w);
            kahan(Sx, cx, a.w * (a.x - r.x));
            kahan(Sy, cy, a.w * (a.y - r.y));
            kahan(Sz, cz, a.w * (a.z - r.z));
        }
        M = row_sum(M - cM);
        cm = make_float3(r.x + row_sum(Sx - cx) / M, r.y + row_sum(Sy - cy) / M, r.z + row_sum(Sz - cz) / M);
        for (int p = nd.x + sub; p < nd.x + nd.y; p += MOM_ROW) {
            const float4 a = pp[p];
            const float dx = a.x - cm.x, dy = a.y - cm.y, dz = a.z - cm.z;
            kahan(Q[0], cQ[0], a.w * dx * dx);
            kahan(Q[1], cQ[1], a.w * dy * dy);
            kahan(Q[2], cQ[2], a.w * dz * dz);
            kahan(Q[3], cQ[3], a.w * dx * dy);
            kahan(Q[4], cQ[4], a.w * dx * dz);
            kahan(Q[5], cQ[5], a.w * dy * dz);
            r2max = fmaxf(r2max, dx * dx + dy * dy + dz * dz);
        }
    } else {
        // lane c < nch takes child c
        const bool has = sub < nch;
        const size_t cv = (size_t)nd.z + (has ? sub : 0);
        nd.y = row_sum(has ? link[cv].y : 0);
        nd.w = nch;
        const float4 r = geo[nd.z];
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b0 = a, b1 = a;
        float rc = 0.f;
        if (has) {
            a = geo[cv];
            b0 = q0[cv];
            b1 = q1[cv];
            rc = a.w;    // the child's rmax
            a.w = b1.w;  // and mass
        }
        M = row_sum(a.w);
        cm = make_float3(r.x + row_sum(a.w * (a.x - r.x)) / M, r.y + row_sum(a.w * (a.y - r.y)) / M,
                         r.z + row_sum(a.w * (a.z - r.z)) / M);
        if (has) {
            const float dx = a.x - cm.x, dy = a.y - cm.y, dz = a.z - cm.z;
            Q[0] = b0.x + a.w * dx * dx;
            Q[1] = b0.y + a.w * dy * dy;
            Q[2] = b0.z + a.w * dz * dz;
            Q[3] = b0.w + a.w * dx * dy;
            Q[4] = b1.x + a.w * dx * dz;
            Q[5] = b1.y + a.w * dy * dz;
            rbound = sqrtf(dx * dx + dy * dy + dz * dz) + rc;
        }
        rbound = row_max(rbound);
        if (nd.y <= RMAX_EXACT_MAX) {
            for (int p = nd.x + sub; p < nd.x + nd.y; p += MOM_ROW) {
                const float4 s = pp[p];
                const float dx = s.x - cm.x, dy = s.y - cm.y, dz = s.z - cm.z;
                r2max = fmaxf(r2max, dx * dx + dy * dy + dz * dz);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 6; k++) Q[k] = row_sum(Q[k] - cQ[k]);
    r2max = row_max(r2max);
    if (sub == 0) {
        const float rmax = nch == 0 || nd.y <= RMAX_EXACT_MAX ? sqrtf(r2max) : rbound;
        // the opening test reads centre and size in one load; the quadrupole goes with the mass and half
        // the trace (the walk's table holds the trace term's line doubled)
        geo[r8] = make_float4(cm.x, cm.y, cm.z, rmax);
        q0[r8] = make_float4(Q[0], Q[1], Q[2], Q[3]);
        q1[r8] = make_float4(Q[4], Q[5], 0.5f * (Q[0] + Q[1] + Q[2]), M);
        if (nch) link[r8] = nd;
    }
}

constexpr int LEVEL_BLOCKS = 2048;  // grid of the per-level launches (grid-stride over the level)
__global__ void moments_f32_kernel(const float4* __restrict__ pp, const uint32_t* __restrict__ dsz, int level,
                                   const int* __restrict__ lev, int4* __restrict__ link, float4* __restrict__ geo,
                                   float4* __restrict__ q0, float4* __restrict__ q1) {
    if (dsz[DSZ_OVERFLOW]) return;
    const uint32_t n = dsz[DSZ_LVL + level], o = dsz[DSZ_LOFF + level];
    const uint32_t end = level < LAGPM_KEY_BITS ? o + n + dsz[DSZ_LVL + level + 1] : o + n;
    const int sub = (int)(threadIdx.x & (MOM_ROW - 1));
    // a record's lanes share i, so they are active or done together and their shuffles stay among them
    for (size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) / MOM_ROW; i < n;
         i += (size_t)gridDim.x * blockDim.x / MOM_ROW)
        moments_f32_node(o + i, sub, end, pp, lev, link, geo, q0, q1);
}
// Levels `bottom` up to `top` in one launch of one workgroup, a barrier between levels: those below the
// expected depth, mostly without a record.
constexpr int MOM_DEEP_THREADS = 1024;
template <typename F>
__device__ inline void moments_deep(const uint32_t* __restrict__ dsz, int bottom, int top, F&& node) {
    if (dsz[DSZ_OVERFLOW]) return;
    for (int l = bottom; l >= top; l--) {
        const uint32_t n = dsz[DSZ_LVL + l], o = dsz[DSZ_LOFF + l];
        if (n == 0) continue;  // the same for every thread
        const uint32_t end = l < LAGPM_KEY_BITS ? o + n + dsz[DSZ_LVL + l + 1] : o + n;
        for (uint32_t i = threadIdx.x / MOM_ROW; i < n; i += MOM_DEEP_THREADS / MOM_ROW)
            node((size_t)(o + i), (int)(threadIdx.x & (MOM_ROW - 1)), end);
        __syncthreads();
    }
}
__global__ void __launch_bounds__(MOM_DEEP_THREADS) moments_f32_deep_kernel(const float4* __restrict__ pp, const uint32_t* __restrict__ dsz,
                                                                            int bottom, int top, const int* __restrict__ lev,
                                                                            int4* link, float4* geo, float4* q0, float4* q1) {
    moments_deep(dsz, bottom, top,
                 [&](size_t r, int sub, uint32_t end) { moments_f32_node(r, sub, end, pp, lev, link, geo, q0, q1); });
}

// FP64 moments for the FP64 path (12 doubles per record), the same way.
__device__ inline double row_sum(double v) {
#pragma unroll
    for (int o = MOM_ROW / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, MOM_ROW);
    return v;
}
__device__ inline double row_max(double v) {
#pragma unroll
    for (int o = MOM_ROW / 2; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, MOM_ROW));
    return v;
}
__device__ inline void moments_f64_node(size_t r8, int sub, uint32_t level_end, const double* __restrict__ x,
                                        const double* __restrict__ y, const double* __restrict__ z, const int* __restrict__ lev,
                                        int4* __restrict__ link, double* __restrict__ nd_d) {
    int4 nd = link[r8];
    const int nch = row_children(lev, nd.z, sub, level_end);
    double M, Q[6] = {0, 0, 0, 0, 0, 0}, rmax = 0, cx, cy, cz;
    if (nch == 0) {
        const double rx = x[nd.x], ry = y[nd.x], rz = z[nd.x];
        double Sx = 0, Sy = 0, Sz = 0;
        for (int p = nd.x + sub; p < nd.x + nd.y; p += MOM_ROW) { Sx += x[p] - rx; Sy += y[p] - ry; Sz += z[p] - rz; }
        M = (double)nd.y;
        cx = rx + row_sum(Sx) / M; cy = ry + row_sum(Sy) / M; cz = rz + row_sum(Sz) / M;
        for (int p = nd.x + sub; p < nd.x + nd.y; p += MOM_ROW) {
            const double dx = x[p] - cx, dy = y[p] - cy, dz = z[p] - cz;
            Q[0] += dx * dx; Q[1] += dy * dy; Q[2] += dz * dz;
            Q[3] += dx * dy; Q[4] += dx * dz; Q[5] += dy * dz;
            rmax = fmax(rmax, dx * dx + dy * dy + dz * dz);
        }
        rmax = sqrt(rmax);
    } else {
        const bool has = sub < nch;
        const size_t cv = (size_t)nd.z + (has ? sub : 0);
        nd.y = row_sum(has ? link[cv].y : 0);
        nd.w = nch;
        const double *a = nd_d + 12 * cv, *r = nd_d + 12 * (size_t)nd.z;
        const double m = has ? a[3] : 0.0, rx = r[0], ry = r[1], rz = r[2];
        M = row_sum(m);
        cx = rx + row_sum(m * (a[0] - rx)) / M; cy = ry + row_sum(m * (a[1] - ry)) / M; cz = rz + row_sum(m * (a[2] - rz)) / M;
        if (has) {
            const double dx = a[0] - cx, dy = a[1] - cy, dz = a[2] - cz;
            Q[0] = a[4] + m * dx * dx; Q[1] = a[5] + m * dy * dy; Q[2] = a[6] + m * dz * dz;
            Q[3] = a[7] + m * dx * dy; Q[4] = a[8] + m * dx * dz; Q[5] = a[9] + m * dy * dz;
            rmax = sqrt(dx * dx + dy * dy + dz * dz) + a[11];
        }
        if (nd.y <= RMAX_EXACT_MAX) {
            double r2 = 0;
            for (int p = nd.x + sub; p < nd.x + nd.y; p += MOM_ROW) {
                const double dx = x[p] - cx, dy = y[p] - cy, dz = z[p] - cz;
                r2 = fmax(r2, dx * dx + dy * dy + dz * dz);
            }
            rmax = sqrt(r2);
        }
    }
#pragma unroll
    for (int k = 0; k < 6; k++) Q[k] = row_sum(Q[k]);
    rmax = row_max(rmax);
    if (sub == 0) {
        double* o = nd_d + 12 * r8;
        o[0] = cx; o[1] = cy; o[2] = cz; o[3] = M;
        for (int k = 0; k < 6; k++) o[4 + k] = Q[k];
        o[10] = Q[0] + Q[1] + Q[2];
        o[11] = rmax;
        if (nch) link[r8] = nd;
    }
}
__global__ void moments_f64_kernel(const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
                                   const uint32_t* __restrict__ dsz, int level, const int* __restrict__ lev,
                                   int4* __restrict__ link, double* __restrict__ nd_d) {
    if (dsz[DSZ_OVERFLOW]) return;
    const uint32_t n = dsz[DSZ_LVL + level], o = dsz[DSZ_LOFF + level];
    const uint32_t end = level < LAGPM_KEY_BITS ? o + n + dsz[DSZ_LVL + level + 1] : o + n;
    const int sub = (int)(threadIdx.x & (MOM_ROW - 1));
    for (size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) / MOM_ROW; i < n;
         i += (size_t)gridDim.x * blockDim.x / MOM_ROW)
        moments_f64_node(o + i, sub, end, x, y, z, lev, link, nd_d);
}

__global__ void __launch_bounds__(MOM_DEEP_THREADS) moments_f64_deep_kernel(const double* __restrict__ x, const double* __restrict__ y,
                                                                            const double* __restrict__ z, const uint32_t* __restrict__ dsz,
                                                                            int bottom, int top, const int* __restrict__ lev, int4* link,
                                                                            double* nd_d) {
    moments_deep(dsz, bottom, top, [&](size_t r, int sub, uint32_t end) { moments_f64_node(r, sub, end, x, y, z, lev, link, nd_d); });
}

// Target groups. A node of at most G particles whose parent holds more than G is a group, as is
// a cell root of at most G; a leaf of more than G (coincident particles) splits into chunks of G.
// Consecutive sibling groups are merged while their sum stays <= G: a parent of more than G packs
// its small children, in order, into runs of contiguous particles. The children of a perturbed
// lattice or a halo are uneven (many of a few particles each), so merging cuts the number of
// groups, and with it of tree walks, to about half while keeping each group inside its parent.
// The parent (or the big leaf, or the small cell root) owns its groups; group_pack visits them.
// Run groups (runs == 1): a chaining cell's particles, in their Morton order, are cut into
// consecutive runs of G (the last one shorter), whatever the tree below the cell: every group but
// the last of a cell fills a wavefront.
// Packed groups (runs == 2): tree groups, except that the small children of a parent are packed
// into runs of exactly G consecutive particles (a run may end inside a child), so the runs of a
// parent fill their wavefronts but the last, and each still lies inside its parent.
template <typename F>
__device__ inline uint32_t group_pack(const int4& nd, int level, int L, int G, int runs, const int4* __restrict__ link, F&& emit) {
    const bool packed = runs == 2;
    if (runs == 1) {
        if (level != L) return 0u;
        const uint32_t c = (uint32_t)((nd.y + G - 1) / G);
        for (uint32_t t = 0; t < c; t++) {
            const int b = nd.x + (int)t * G;
            emit(b, min(nd.x + nd.y, b + G) - b);
        }
        return c;
    }
    if (nd.y <= G) {
        if (level != L) return 0u;  // a small node below the cell level belongs to its parent's runs
        emit(nd.x, nd.y);
        return 1u;
    }
    if (nd.w == 0) {
        const uint32_t c = (uint32_t)((nd.y + G - 1) / G);
        for (uint32_t t = 0; t < c; t++) {
            const int b = nd.x + (int)t * G;
            emit(b, min(nd.x + nd.y, b + G) - b);
        }
        return c;
    }
    uint32_t c = 0;
    int rb = 0, rn = 0;  // the open run: first particle, count
    for (int k = 0; k < nd.w; k++) {
        const int4 ci = link[nd.z + k];
        if (ci.y > G) {  // a big child owns its own groups and ends the run
            if (rn) { emit(rb, rn); c++; rn = 0; }
            continue;
        }
        if (packed) {  // the run takes the child's particles and is cut at exactly G
            if (!rn) rb = ci.x;
            rn += ci.y;
            while (rn >= G) { emit(rb, G); c++; rb += G; rn -= G; }
            continue;
        }
        if (rn && rn + ci.y > G) { emit(rb, rn); c++; rn = 0; }
        if (!rn) rb = ci.x;
        rn += ci.y;
    }
    if (rn) { emit(rb, rn); c++; }
    return c;
}
// Groups in the nodes' pre-order (so neighbouring groups are near in space): counts per block of
// GB_NODES nodes, a scan of the blocks' counts, and the groups themselves. Blocks past the node count
// leave at once.
constexpr int GB_THREADS = 256;
constexpr int GB_ITEMS = 4;
constexpr int GB_NODES = GB_THREADS * GB_ITEMS;
__global__ void __launch_bounds__(GB_THREADS) group_count_kernel(const uint32_t* __restrict__ dsz, size_t cap, int L, int G, int runs,
                                                                 const int4* __restrict__ link, const int* __restrict__ lev,
                                                                 const uint32_t* __restrict__ rop, uint32_t* __restrict__ gcnt) {
    __shared__ uint32_t sum;
    const size_t n = dsz[DSZ_OVERFLOW] ? 0 : dev_count(dsz, DSZ_NODES, cap), first = (size_t)blockIdx.x * GB_NODES;
    if (first >= n) {
        if (threadIdx.x == 0) gcnt[blockIdx.x] = 0u;
        return;
    }
    if (threadIdx.x == 0) sum = 0u;
    __syncthreads();
    uint32_t c = 0u;
#pragma unroll
    for (int q = 0; q < GB_ITEMS; q++) {
        const size_t v = first + (size_t)q * GB_THREADS + threadIdx.x;
        if (v < n) {
            const uint32_t r = rop[v];
            c += group_pack(link[r], lev[r] & 255, L, G, runs, link, [](int, int) {});
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += (uint32_t)__shfl_xor((int)c, o, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(&sum, c);
    __syncthreads();
    if (threadIdx.x == 0) gcnt[blockIdx.x] = sum;
}
__global__ void __launch_bounds__(256) group_rows_kernel(const uint32_t* __restrict__ gcnt, uint32_t* __restrict__ goff, uint32_t nblk,
                                                         size_t gcap, uint32_t* __restrict__ dsz) {
    const uint32_t total = block_row_scan(gcnt, goff, nblk);
    if (threadIdx.x == 0) {
        dsz[DSZ_GROUPS] = total;
        if (total > gcap) dsz[DSZ_OVERFLOW] = 1u;
    }
}
__global__ void __launch_bounds__(GB_THREADS) group_write_kernel(const uint32_t* __restrict__ dsz, size_t cap, int L, int G, int runs,
                                                                 const int4* __restrict__ link, const int* __restrict__ lev,
                                                                 const uint32_t* __restrict__ rop, const uint32_t* __restrict__ goff,
                                                                 int2* __restrict__ groups) {
    __shared__ uint32_t wsum[GB_NODES / 64];
    const size_t n = dsz[DSZ_OVERFLOW] ? 0 : dev_count(dsz, DSZ_NODES, cap), first = (size_t)blockIdx.x * GB_NODES;
    if (first >= n) return;
    const int lane = (int)(threadIdx.x & 63), wid = (int)(threadIdx.x >> 6);
    int4 nd[GB_ITEMS];
    int level[GB_ITEMS];
    uint32_t at[GB_ITEMS];
#pragma unroll
    for (int q = 0; q < GB_ITEMS; q++) {
        const size_t v = first + (size_t)q * GB_THREADS + threadIdx.x;
        uint32_t c = 0u;
        nd[q] = make_int4(0, 0, 0, 0);
        if (v < n) {
            const uint32_t r = rop[v];
            nd[q] = link[r];
            level[q] = lev[r] & 255;
            c = group_pack(nd[q], level[q], L, G, runs, link, [](int, int) {});
        }
        int wt;
        at[q] = (uint32_t)wave_excl_scan((int)c, lane, wt);
        if (!c) nd[q].y = 0;
        if (lane == 0) wsum[q * (GB_THREADS / 64) + wid] = (uint32_t)wt;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < GB_ITEMS; q++) {
        if (!nd[q].y) continue;
        uint32_t g = goff[blockIdx.x] + at[q];
        for (int w = 0; w < q * (GB_THREADS / 64) + wid; w++) g += wsum[w];
        group_pack(nd[q], level[q], L, G, runs, link, [&](int b, int m) { groups[g++] = make_int2(b, m); });
    }
}

// an empty box's tree: clear the size words and the interaction counters
__global__ void tree_reset_kernel(uint32_t* __restrict__ dsz, unsigned long long* __restrict__ counters) {
    tree_reset(threadIdx.x, dsz, counters);
}

// ---------------------------------------------------------------------------------------
// Walk helpers
template <int V>
struct ic {  // a compile-time int for generic lambdas
    static constexpr int value = V;
};

__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// periodic image offset of neighbour nb (0..26) of cell (cx,cy,cz)
__device__ inline float image_shift(int c, int d, int mcell, float box) {
    int t = c + d;
    return t < 0 ? -box : (t >= mcell ? box : 0.0f);
}

}  // namespace

// Device view of one box for the walk. The force tables are per unit n^2 (shared by boxes of
// equal law, softening and split), so `fact` carries the box's kick factor times 1/n^2.
struct walk_box {
    const float4* pp;
    // the tree by record (the build's order: the children of a node are consecutive records)
    const int4* link;      // first particle, count, first child record, children
    const float4* geo;     // com, rmax
    const float4* q0;      // Qxx Qyy Qzz Qxy
    const float4* q1;      // Qxz Qyz trQ, mass
    const int* cellroot;   // root record of each chaining cell, or -1
    const int2* groups;
    const uint64_t* key;
    double *tvx, *tvy, *tvz;       // the tree kick of each particle (written, not added: see below)
    unsigned long long* counters;  // [0] n_pp, [1] n_pc, [2] walk stack overflow
    uint32_t* dsz;                 // sizes; the walk sets DSZ_WALKOVF on a stack overflow
    int cell_shift;
    int mcell;
    int naccept;
    float box;       // n
    float rc2;
    float rcut;
    float inv_theta2;
    float fact;
};

namespace {

// Group prefix over the boxes of one walk launch (a box whose build overflowed contributes no
// groups and so gets no kick) and the reset of the group tickets (one per XCD range).
__global__ void walk_prefix_kernel(const walk_box* __restrict__ B, int nbox, uint32_t* __restrict__ prefix,
                                   unsigned* __restrict__ ticket) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    uint32_t s = 0;
    for (int b = 0; b < nbox; b++) {
        prefix[b] = s;
        const uint32_t* d = B[b].dsz;
        s += d[DSZ_OVERFLOW] ? 0u : d[DSZ_GROUPS];
    }
    prefix[nbox] = s;
    for (int x = 0; x < WALK_XCDS; x++) ticket[x * LAGPM_TICKET_STRIDE] = 0u;
}

// CENSUS: also count the evaluated particle pairs that lie within the cutoff (counters[3]), a
// measurement of the lists' useful fraction; it adds a compare and an add per pair.
// Pointers read from a descriptor in memory are generic to the compiler, which then emits flat
// loads and stores. A flat access also counts against the LDS wait counter, so every LDS wait that
// follows one waits for the memory access too; these casts make them global ones.
template <typename T>
__device__ inline const __attribute__((address_space(1))) T* gld(const T* p) {
    return (const __attribute__((address_space(1))) T*)p;
}
template <typename T>
__device__ inline __attribute__((address_space(1))) T* gst(T* p) {
    return (__attribute__((address_space(1))) T*)p;
}
// (the HIP vector types do not copy from a global reference: load as clang vectors)
typedef float gv4f __attribute__((ext_vector_type(4)));
typedef int gv4i __attribute__((ext_vector_type(4)));
typedef int gv2i __attribute__((ext_vector_type(2)));
__device__ inline float4 gld4(const float4* p, size_t i) {
    const gv4f v = ((const __attribute__((address_space(1))) gv4f*)p)[i];
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ inline int4 gld4(const int4* p, size_t i) {
    const gv4i v = ((const __attribute__((address_space(1))) gv4i*)p)[i];
    return make_int4(v.x, v.y, v.z, v.w);
}
__device__ inline int2 gld2(const int2* p, size_t i) {
    const gv2i v = ((const __attribute__((address_space(1))) gv2i*)p)[i];
    return make_int2(v.x, v.y);
}

template <bool LOGT, bool CENSUS>
__global__ void __launch_bounds__(WALK_THREADS) walk_f32_kernel(const walk_box* __restrict__ B, const uint32_t* __restrict__ gprefix,
                                                                int nbox, const float2* __restrict__ tab0,
                                                                const float4* __restrict__ tab12, int* __restrict__ stacks,
                                                                unsigned* __restrict__ ticket_ctr) {
    // positions are in scaled units (tree_count_kernel): for the log tables r^2 here is lam r^2
    constexpr float lam = 1.0f;
    // One 1024-thread workgroup per CU: the 16 waves share one LDS copy of the particle force
    // table (32 KB) next to their private interaction lists.
    __shared__ float2 s_tab0[TAB_LDS];
    __shared__ uint32_t s_ppidx[WALK_WAVES][PP_CAP];
    __shared__ int s_stack[WALK_WAVES][LSTACK > 0 ? LSTACK : 1];
    __shared__ int s_pcidx[WALK_WAVES][PC_CAP];
    // Staged particles need three words (their masses are 1) and a node's third record three (its
    // fourth is the mass, kept beside the centre). With the log tables the LDS pipe is the bound
    // (90 % busy at 256^3) and 12-byte entries take fewer of its cycles than 16-byte ones: walk
    // 12.95 -> 12.55 ms at 256^3. The reference law is bound by its arithmetic (3.76 -> 3.90 ms with
    // 12 bytes) and keeps 16.
    using psrc = std::conditional_t<LOGT, float3, float4>;
    __shared__ psrc s_pp[WALK_WAVES][64];
    __shared__ float4 s_pc[WALK_WAVES][2][64];
    __shared__ psrc s_pc2[WALK_WAVES][64];
    __shared__ float4 s_shift[WALK_WAVES][27];  // the group's image shift of each neighbour cell
    __shared__ unsigned s_done;  // bit x: range x was found exhausted by a wave of this workgroup
    if (threadIdx.x == 0) s_done = 0u;
    constexpr int NBIN = LOGT ? LAGPM_LOG_BINS : 4096;
    for (int i = threadIdx.x; i < NBIN; i += WALK_THREADS) s_tab0[i] = tab0[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t* ppidx = s_ppidx[wid];
    int* pcidx = s_pcidx[wid];
    psrc* cpp = s_pp[wid];
    float4* cpc0 = s_pc[wid][0];
    float4* cpc1 = s_pc[wid][1];
    psrc* cpc2 = s_pc2[wid];
    int* gstack = stacks + (size_t)(blockIdx.x * WALK_WAVES + wid) * STACK_MAX;
    int* lstack = s_stack[wid];
    // stack entry i: LDS below LSTACK (96% of pop rounds stay there), global memory above
    // (the LDS read is unconditional, from a clamped index, so that the compiler does not merge
    // the two reads into one flat load through a selected pointer: a flat load also holds up every
    // LDS wait behind it)
    auto sget = [&](int i) -> int {
        const int l = lstack[i < LSTACK ? i : LSTACK - 1];
        int g = 0;
        if (i >= LSTACK) g = gstack[i];
        return i < LSTACK ? l : g;
    };
    auto sset = [&](int i, int v) {
        if (i < LSTACK) lstack[i] = v;
        else gstack[i] = v;
    };
    const int gtotal = __builtin_amdgcn_readfirstlane((int)gprefix[nbox]);
    // XCD-local group ranges. Workgroups are dispatched to the XCDs round robin (block b runs on
    // XCD b % 8), and each XCD has its own L2. The groups are in Morton order, so giving XCD x
    // the contiguous range x of 8 keeps the sources and nodes that neighbouring groups share in
    // one L2; a single global ticket would spread neighbours over all eight caches. An XCD that
    // has finished its range takes tickets from the next ranges in turn (work stealing), and a
    // wave leaves after finding all eight ranges exhausted.
    // A wave's first group of its own range is its rank there (the waves of one workgroup far apart, so
    // that few groups spread over all CUs), without an atomic. Later ones come from the range's
    // counter, each counter in a cache line of its own. Once a range is found exhausted the workgroup's
    // other waves skip it, and a range that the ranks alone cover is never asked for. Device-wide
    // atomics on one line are served one after another: when every wave began with one and left by
    // asking all eight ranges (33,000 atomics for the 741 groups of a 32^3 box), their queue held up
    // the first loads of the waves that had a group by 0.2 ms of a 0.63 ms walk. Spreading a
    // workgroup's first groups took 0.1 more. Walk in ms before and after: 32^3 0.63 -> 0.30, 64^3
    // 0.75 -> 0.59, 100^3 1.47 -> 1.30, 128^3 2.14 -> 1.91, 256^3 13.94 -> 13.75.
    auto range_lo = [&](int x) -> int { return (int)(((long long)gtotal * x) / WALK_XCDS); };
    auto range_waves = [&](int x) -> int { return (((int)gridDim.x - x + WALK_XCDS - 1) / WALK_XCDS) * WALK_WAVES; };
    const int home = (int)(blockIdx.x % WALK_XCDS);
    int tries = -1;  // ranges found exhausted; -1: the rank is still to be taken

    for (;;) {
        const int slot = (home + max(tries, 0)) % WALK_XCDS;
        const int lo = range_lo(slot), left = range_lo(slot + 1) - lo, ranked = range_waves(slot);
        int t = left;
        if (tries < 0) {
            t = __builtin_amdgcn_readfirstlane(wid) * (ranked / WALK_WAVES) + (int)(blockIdx.x / WALK_XCDS);
            tries = 0;
        } else if (left > ranked && !((__builtin_amdgcn_readfirstlane((int)*(volatile unsigned*)&s_done) >> slot) & 1)) {
            // Group ticket: one atomic per group, from lane 0 (an atomic executed by all 64 lanes is
            // 64 serialised operations on one address, which capped the group rate). The ticket is
            // then read from lane 0 into a scalar register, so every branch of the loop below is
            // wave-uniform: the compiler cannot thread the back edge differently per lane (which
            // would let lanes 1..63 re-enter a group without a new ticket). A counter passes its
            // range's size by at most one per wave, so its low word holds it.
            unsigned ticket = 0u;
            if (lane == 0) ticket = atomicAdd(ticket_ctr + slot * LAGPM_TICKET_STRIDE, 1u);
            t = ranked + __builtin_amdgcn_readlane((int)ticket, 0);
            if (t >= left && lane == 0) atomicOr(&s_done, 1u << slot);
        }
        if (t >= left) {
            if (++tries == WALK_XCDS) break;
            continue;
        }
        const int g = lo + t;
        // the box that owns global group g: largest b with gprefix[b] <= g (wave-uniform search)
        int blo = 0, bhi = nbox;
        while (bhi - blo > 1) {
            const int mid = (blo + bhi) >> 1;
            if (__builtin_amdgcn_readfirstlane((int)gprefix[mid]) <= g) blo = mid;
            else bhi = mid;
        }
        const walk_box A = B[blo];
        const int2 gr = gld2(A.groups, g - __builtin_amdgcn_readfirstlane((int)gprefix[blo]));
        const int cnt = __builtin_amdgcn_readfirstlane(gr.y);
        const int gbeg = __builtin_amdgcn_readfirstlane(gr.x);
        // Lane layout. Lane (tgt, rep) holds M targets, tgt + i Tw for i < M, and takes every R-th
        // source of a chunk from rep on; the R partial sums of a target are added at the end.
        // With M = 1, R = 64/Tw lanes per target, Tw the smallest power of two >= cnt, the lanes
        // past cnt idle: for 33-48 targets a third of the wave or more. M = 3 targets per lane
        // fill ceil(cnt/3) slots instead, and each staged source or node is read once for three
        // targets. A group takes M = 3 where it uses at least 4/3 of the lanes M = 1 would
        // (cnt in 33-48, 17-24, 9-12, 5-6), and for 65-192 targets, which one target per lane
        // cannot hold. (Two and five targets per lane as well, for the remaining gaps, made the
        // kernel's code four times larger and spilled registers: the walk got slower.)
        int R = 1;
        while (cnt * 2 * R <= 64) R <<= 1;
        int M = 1;
        {
            const int s3 = (cnt + 2) / 3;
            int R3 = 1;
            while (s3 * 2 * R3 <= 64) R3 <<= 1;
            if (cnt > 64 || R3 >= 4 * R) {
                M = 3;
                R = R3;
            }
        }
        const int Tw = 64 / R;
        const int tgt = lane & (Tw - 1), rep = lane / Tw;
        const uint64_t cellkey = gld(A.key)[gbeg] >> A.cell_shift;
        const int cx = (int)compact3(cellkey), cy = (int)compact3(cellkey >> 1), cz = (int)compact3(cellkey >> 2);
        // the rest of the group, compiled once per targets-per-lane count so that the single-target
        // path carries no registers for the other two
        auto group_body = [&](auto mc) {
        constexpr int M = decltype(mc)::value;
        bool valid[M];
        int me[M];
        float4 xt[M];
        float ax[M], ay[M], az[M];
        float lx = 0.f, ly = 0.f, lz = 0.f, hx = 0.f, hy = 0.f, hz = 0.f;
#pragma unroll
        for (int i = 0; i < M; i++) {
            const int t = tgt + i * Tw;
            valid[i] = t < cnt;
            me[i] = gbeg + (valid[i] ? t : 0);  // an idle slot repeats target 0: inside the group box
            xt[i] = gld4(A.pp, me[i]);
            ax[i] = ay[i] = az[i] = 0.f;
            lx = i ? fminf(lx, xt[i].x) : xt[i].x; hx = i ? fmaxf(hx, xt[i].x) : xt[i].x;
            ly = i ? fminf(ly, xt[i].y) : xt[i].y; hy = i ? fmaxf(hy, xt[i].y) : xt[i].y;
            lz = i ? fminf(lz, xt[i].z) : xt[i].z; hz = i ? fmaxf(hz, xt[i].z) : xt[i].z;
        }
        const float lox = wave_minf(lx), loy = wave_minf(ly), loz = wave_minf(lz);
        const float hix = wave_maxf(hx), hiy = wave_maxf(hy), hiz = wave_maxf(hz);
        unsigned long long npp = 0, npc = 0;
        unsigned nin = 0;  // CENSUS: this lane's pairs within the cutoff
        int sp = 0;
        bool overflow = false;
        {
            int e = -1;
            if (lane < 27) {
                int dx = lane % 3 - 1, dy = (lane / 3) % 3 - 1, dz = lane / 9 - 1;
                int nx = (cx + dx + A.mcell) % A.mcell, ny = (cy + dy + A.mcell) % A.mcell, nz = (cz + dz + A.mcell) % A.mcell;
                int r = gld(A.cellroot)[nx + A.mcell * (ny + A.mcell * nz)];
                if (r >= 0) e = (r << 5) | lane;
            }
            int tot;
            int off = wave_excl_count(e >= 0, tot);
            if (e >= 0) sset(off, e);
            sp = tot;
        }
        int pp_n = 0, pc_n = 0;

        // The periodic image shift of each of the 27 neighbour cells, made once per group (lane nb
        // makes entry nb) and then read from LDS: a lookup, where computing it (three compares and
        // selects per axis and the base-3 digits of nb) cost some 25 operations per use, and every
        // staged particle, staged node and popped node uses one.
        if (lane < 27)
            s_shift[wid][lane] = make_float4(image_shift(cx, lane % 3 - 1, A.mcell, A.box),
                                             image_shift(cy, (lane / 3) % 3 - 1, A.mcell, A.box),
                                             image_shift(cz, lane / 9 - 1, A.mcell, A.box), 0.f);
        wave_sync();
        auto shift_of = [&](int nb, float& sx, float& sy, float& sz) {
            const float4 sh = s_shift[wid][nb];
            sx = sh.x;
            sy = sh.y;
            sz = sh.z;
        };
        // Source chunks are staged in LDS; entries past m are far-away
        // dummies of zero mass, so every lane runs the same unrolled trip count and the cutoff
        // is a select (no branch, no exec-mask loop).
        // (8 box lengths away: sources lie within one box length of [0, n), and n >= 4 cutoffs)
        const float4 dummy = make_float4(8.f * A.box, 8.f * A.box, 8.f * A.box, 0.f);
        auto to_src = [](const float4& q) -> psrc {
            if constexpr (LOGT) return make_float3(q.x, q.y, q.z);
            else return q;
        };
        auto load_pp = [&](int start, int m) -> psrc {
            float4 s = dummy;
            if (lane < m) {
                uint32_t e = ppidx[start + lane];
                float sx, sy, sz;
                shift_of((int)(e & 31u), sx, sy, sz);
                s = gld4(A.pp, e >> 5);
                s.x += sx; s.y += sy; s.z += sz;
            }
            return to_src(s);
        };
        // Pair sums over one staged chunk. Lane (tgt, rep) takes the sources rep, rep + R, ...
        // (neighbouring lanes read neighbouring entries: no LDS bank conflicts). R is a template
        // value here, so the loads of one round are immediate offsets from one address. Sources
        // are taken four at a time: their LDS loads, then their table loads, are issued together
        // so one wave's LDS latency overlaps its own arithmetic.
        auto pp_one = [&](psrc s) {
#pragma unroll
            for (int i = 0; i < M; i++) {
                float dx = xt[i].x - s.x, dy = xt[i].y - s.y, dz = xt[i].z - s.z;
                float r2 = dx * dx + dy * dy + dz * dz;
                if constexpr (CENSUS) nin += (valid[i] && r2 <= A.rc2) ? 1u : 0u;
                float t;
                const int nt = table_bin<LOGT>(r2, t, lam);
                float2 tb = s_tab0[nt];
                float f = tb.x + tb.y * t;  // particle masses are 1 here: the box mass is in fact
                if constexpr (!LOGT) f = (r2 <= A.rc2) ? f : 0.f;
                ax[i] += dx * f; ay[i] += dy * f; az[i] += dz * f;
            }
        };
        auto pp_chunk_r = [&](auto rc) {
            constexpr int RR = decltype(rc)::value;
            constexpr int iters = 64 / RR;
            constexpr int U = M == 1 ? 4 : 2;  // sources per round: U M pairs in flight
            const psrc* src = cpp + rep;
            if constexpr (LOGT && M == 1 && iters >= 2 * U) {
                // Two rounds in flight: while a round's table lines and the sources after it are on their
                // way, the round before is added up. Where a walk lasts as long as its heaviest group, a wave
                // by itself on its SIMD waits for every LDS read otherwise: 41 ns a source, of which 20
                // are the issue of its operations. Walk 32^3 theta 0 0.61 -> 0.56 ms, 64^3
                // 0.59 -> 0.56, 32^3 0.306 -> 0.293; with 16 waves a CU (256^3) 12.9 either way. Eight
                // sources a round spill (256^3 28 ms), two gain nothing, three targets a lane neither (their
                // rounds have six pairs). The fused operations are written out: the same bits as the plain loop.
                constexpr int NB = iters / U;  // rounds, an even number
                struct round {
                    float dx[U], dy[U], dz[U], r2[U];
                    float2 tb[U];
                } P, Q;
                psrc s[U];
                auto load = [&](int b) {
#pragma unroll
                    for (int u = 0; u < U; u++) s[u] = src[(b * U + u) * RR];
                };
                auto diff = [&](round& B) {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        B.dx[u] = xt[0].x - s[u].x; B.dy[u] = xt[0].y - s[u].y; B.dz[u] = xt[0].z - s[u].z;
                    }
                };
                auto look = [&](round& B) {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        B.r2[u] = fmaf(B.dz[u], B.dz[u], fmaf(B.dx[u], B.dx[u], B.dy[u] * B.dy[u]));
                        if constexpr (CENSUS) nin += (valid[0] && B.r2[u] <= A.rc2) ? 1u : 0u;
                        float t;
                        B.tb[u] = s_tab0[table_bin<LOGT>(B.r2[u], t, lam)];
                    }
                };
                auto add = [&](const round& B) {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const float f = fmaf(B.tb[u].y, B.r2[u], B.tb[u].x);
                        ax[0] = fmaf(B.dx[u], f, ax[0]); ay[0] = fmaf(B.dy[u], f, ay[0]); az[0] = fmaf(B.dz[u], f, az[0]);
                    }
                };
                load(0);
                diff(P);
                load(1);
                look(P);
#pragma unroll 1
                for (int b = 1; b + 1 < NB; b += 2) {
                    diff(Q);
                    load(b + 1);
                    look(Q);
                    add(P);
                    diff(P);
                    load(b + 2);
                    look(P);
                    add(Q);
                }
                diff(Q);
                look(Q);
                add(P);
                add(Q);
            } else if constexpr (iters >= U) {
#pragma unroll 2
                for (int k = 0; k < iters; k += U) {
                    psrc s[U];
                    float dx[U][M], dy[U][M], dz[U][M], r2[U][M];
                    bool any = false;
#pragma unroll
                    for (int u = 0; u < U; u++) s[u] = src[(k + u) * RR];
#pragma unroll
                    for (int u = 0; u < U; u++)
#pragma unroll
                        for (int i = 0; i < M; i++) {
                            dx[u][i] = xt[i].x - s[u].x; dy[u][i] = xt[i].y - s[u].y; dz[u][i] = xt[i].z - s[u].z;
                            r2[u][i] = dx[u][i] * dx[u][i] + dy[u][i] * dy[u][i] + dz[u][i] * dz[u][i];
                            if constexpr (!LOGT) any = any || (r2[u][i] <= A.rc2);
                            if constexpr (CENSUS) nin += (valid[i] && r2[u][i] <= A.rc2) ? 1u : 0u;
                        }
                    if constexpr (!LOGT)
                        if (!__any(any)) continue;  // wave-uniform skip of U far sources
                    float2 tb[U][M];
                    float t[U][M];
#pragma unroll
                    for (int u = 0; u < U; u++)
#pragma unroll
                        for (int i = 0; i < M; i++) tb[u][i] = s_tab0[table_bin<LOGT>(r2[u][i], t[u][i], lam)];
#pragma unroll
                    for (int u = 0; u < U; u++)
#pragma unroll
                        for (int i = 0; i < M; i++) {
                            float f = tb[u][i].x + tb[u][i].y * t[u][i];
                            if constexpr (!LOGT) f = (r2[u][i] <= A.rc2) ? f : 0.f;
                            ax[i] += dx[u][i] * f; ay[i] += dy[u][i] * f; az[i] += dz[u][i] * f;
                        }
                }
            } else {
#pragma unroll
                for (int k = 0; k < iters; k++) pp_one(src[k * RR]);
            }
        };
        // the common replications take the unrolled loops (one target per lane: groups of more
        // than 8 targets, R <= 4; three: more than 12, R <= 8); the rest a plain loop
        auto pp_chunk = [&]() {
            if (R == 1) pp_chunk_r(ic<1>{});
            else if (R == 2) pp_chunk_r(ic<2>{});
            else if (R == 4) pp_chunk_r(ic<4>{});
            else if (M == 3 && R == 8) pp_chunk_r(ic<8>{});
            else
                for (int k = 0; k < 64 / R; k++) pp_one(cpp[rep + k * R]);
        };
        // flush `nchunk` consecutive chunks starting at list entry `start` (the last may be
        // partial: `mlast` entries); the next chunk's global loads overlap this chunk's math
        // Staging with a cut: a listed particle farther than the cutoff from the group's bounding
        // box is beyond it from every target, so its pair terms are exactly zero (the table is zero
        // there, and the reference law's select zeroes it); it is dropped before it costs a chunk
        // slot. The margin keeps every dropped pair clear of the float-rounded table edge.
        const float rc2_keep = A.rc2 * (1.0f + 1.0e-5f);
        auto near_group = [&](psrc q) -> bool {
            const float ddx = fmaxf(fmaxf(lox - q.x, q.x - hix), 0.f);
            const float ddy = fmaxf(fmaxf(loy - q.y, q.y - hiy), 0.f);
            const float ddz = fmaxf(fmaxf(loz - q.z, q.z - hiz), 0.f);
            return ddx * ddx + ddy * ddy + ddz * ddz <= rc2_keep;
        };
        int fill = 0;  // staged particles in cpp[0, fill), wave-uniform
        // append the kept particles of one 64-entry block to the chunk, computing the chunk when it
        // fills; survivors past its end start the next chunk
        auto stage_pp = [&](psrc q, bool keep) {
            int tot;
            const int off = wave_excl_count(keep, tot);
            const int room = 64 - fill;
            if (keep && off < room) cpp[fill + off] = q;
            if (tot >= room) {
                wave_sync();
                pp_chunk();
                npp += 64ull;
                wave_sync();
                if (keep && off >= room) cpp[off - room] = q;
                fill = tot - room;
            } else {
                fill += tot;
            }
            wave_sync();
        };
        // stage `nblock` consecutive blocks of the list from entry `start` (the last may be
        // partial: `mlast` entries); the next block's global loads overlap this block's chunk
        auto flush_pp = [&](int start, int nblock, int mlast) {
            psrc nxt = load_pp(start, nblock == 1 ? mlast : 64);
            for (int c = 0; c < nblock; c++) {
                const psrc cur = nxt;
                if (c + 1 < nblock) nxt = load_pp(start + 64 * (c + 1), c + 2 == nblock ? mlast : 64);
                stage_pp(cur, near_group(cur));  // entries past m are far dummies: never kept
            }
        };
        // One node interaction: monopole plus quadrupole, Q d computed once and reused for
        // d.Q.d (the quadratic form) and for the 2 f2 Q d term. The table's f2 line is stored
        // doubled and the node's trace halved (both exact), so 2 f2 is the table value itself.
        auto pc_eval = [&](float4 c, float4 qa, psrc qb, float2 t0, float4 t12, float t, float dx, float dy, float dz,
                           bool in, float& ax, float& ay, float& az) {
            float f1 = t0.x + t0.y * t, f2 = t12.x + t12.y * t, f3 = t12.z + t12.w * t;
            float qx1 = qa.x * dx + qa.w * dy + qb.x * dz;
            float qx2 = qa.w * dx + qa.y * dy + qb.y * dz;
            float qx3 = qb.x * dx + qb.y * dy + qa.z * dz;
            float qxy = dx * qx1 + dy * qx2 + dz * qx3;
            float tmp = c.w * f1 + qb.z * f2 + qxy * f3;
            float two = f2;
            if constexpr (!LOGT) {
                tmp = in ? tmp : 0.f;
                two = in ? two : 0.f;
            }
            ax = fmaf(qx1, two, fmaf(dx, tmp, ax));
            ay = fmaf(qx2, two, fmaf(dy, tmp, ay));
            az = fmaf(qx3, two, fmaf(dz, tmp, az));
        };
        // one node against this lane's M targets
        auto pc_node = [&](const float4& c, const float4& qa, const psrc& qb) {
#pragma unroll
            for (int i = 0; i < M; i++) {
                const float dx = xt[i].x - c.x, dy = xt[i].y - c.y, dz = xt[i].z - c.z;
                const float r2 = dx * dx + dy * dy + dz * dz;
                float t;
                const int nt = table_bin<LOGT>(r2, t, lam);
                pc_eval(c, qa, qb, s_tab0[nt], tab12[nt], t, dx, dy, dz, r2 <= A.rc2, ax[i], ay[i], az[i]);
            }
        };
        auto pc_chunk_r = [&](auto rc) {
            constexpr int RR = decltype(rc)::value;
            constexpr int iters = 64 / RR;
            constexpr int U = M == 1 ? 2 : 1;  // nodes per round: U M interactions in flight
            const float4* n0 = cpc0 + rep;
            const float4* n1 = cpc1 + rep;
            const psrc* n2 = cpc2 + rep;
            if constexpr (iters >= 2) {
                // the nodes' loads first, then their table loads, as for the particles
#pragma unroll 2
                for (int k = 0; k < iters; k += U) {
                    float4 c[U], qa[U];
                    psrc qb[U];
                    float dx[U][M], dy[U][M], dz[U][M], r2[U][M];
                    bool any = false;
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const int j = (k + u) * RR;
                        c[u] = n0[j]; qa[u] = n1[j]; qb[u] = n2[j];
                    }
#pragma unroll
                    for (int u = 0; u < U; u++)
#pragma unroll
                        for (int i = 0; i < M; i++) {
                            dx[u][i] = xt[i].x - c[u].x; dy[u][i] = xt[i].y - c[u].y; dz[u][i] = xt[i].z - c[u].z;
                            r2[u][i] = dx[u][i] * dx[u][i] + dy[u][i] * dy[u][i] + dz[u][i] * dz[u][i];
                            if constexpr (!LOGT) any = any || (r2[u][i] <= A.rc2);
                        }
                    if constexpr (!LOGT)
                        if (!__any(any)) continue;  // wave-uniform skip of far nodes
                    float t[U][M];
                    float2 t0[U][M];
                    float4 t12[U][M];
#pragma unroll
                    for (int u = 0; u < U; u++)
#pragma unroll
                        for (int i = 0; i < M; i++) {
                            const int nt = table_bin<LOGT>(r2[u][i], t[u][i], lam);
                            t0[u][i] = s_tab0[nt];
                            t12[u][i] = tab12[nt];
                        }
#pragma unroll
                    for (int u = 0; u < U; u++)
#pragma unroll
                        for (int i = 0; i < M; i++)
                            pc_eval(c[u], qa[u], qb[u], t0[u][i], t12[u][i], t[u][i], dx[u][i], dy[u][i], dz[u][i],
                                    r2[u][i] <= A.rc2, ax[i], ay[i], az[i]);
                }
            } else {
                pc_node(n0[0], n1[0], n2[0]);
            }
        };
        auto flush_pc = [&](int start, int m) {
            if (lane < m) {
                int e = pcidx[start + lane];
                float sx, sy, sz;
                shift_of(e & 31, sx, sy, sz);
                int v = e >> 5;
                const float4 c = gld4(A.geo, v), q1 = gld4(A.q1, v);
                cpc0[lane] = make_float4(c.x + sx, c.y + sy, c.z + sz, q1.w);  // (centre, mass)
                cpc1[lane] = gld4(A.q0, v);
                cpc2[lane] = to_src(q1);
            } else {
                cpc0[lane] = dummy;
                cpc1[lane] = make_float4(0.f, 0.f, 0.f, 0.f);
                cpc2[lane] = to_src(make_float4(0.f, 0.f, 0.f, 0.f));
            }
            wave_sync();
            if (R == 1) pc_chunk_r(ic<1>{});
            else if (R == 2) pc_chunk_r(ic<2>{});
            else if (R == 4) pc_chunk_r(ic<4>{});
            else if (M == 3 && R == 8) pc_chunk_r(ic<8>{});
            else
                for (int k = 0; k < 64 / R; k++) {
                    const int j = rep + k * R;
                    pc_node(cpc0[j], cpc1[j], cpc2[j]);
                }
            npc += (unsigned long long)m;
            wave_sync();
        };

        int iters = 0;
        while (sp > 0) {
            if (++iters > WALK_MAX_ITERS) {  // a well-formed tree never gets here
                overflow = true;
                break;
            }
            const int take = min(sp, 64);
            sp -= take;
            int e = lane < take ? sget(sp + lane) : -1;
            int kind = 0;  // 0 none, 1 accept, 2 leaf, 3 open
            int4 nd = make_int4(0, 0, 0, 0);  // (first particle, count, first child record, children)
            int v = 0, nb = 0;
            if (e >= 0) {
                v = e >> 5;
                nb = e & 31;
                float sx, sy, sz;
                shift_of(nb, sx, sy, sz);
                // two 16-byte loads per node: the children are consecutive records, so opening a
                // node needs only the first one's index, and the popped nodes of a round (mostly
                // the children of the previous round's opened nodes) share cache lines
                const float4 c = gld4(A.geo, v);
                const float rmax = c.w;
                nd = gld4(A.link, v);
                float px = c.x + sx, py = c.y + sy, pz = c.z + sz;
                float ddx = fmaxf(fmaxf(lox - px, px - hix), 0.f);
                float ddy = fmaxf(fmaxf(loy - py, py - hiy), 0.f);
                float ddz = fmaxf(fmaxf(loz - pz, pz - hiz), 0.f);
                float dmin2 = ddx * ddx + ddy * ddy + ddz * ddz;
                float rr = A.rcut + rmax;
                if (dmin2 > rr * rr) kind = 0;
                else if (nd.y >= A.naccept && dmin2 >= rmax * rmax * A.inv_theta2) kind = 1;
                else if (nd.w == 0) kind = 2;
                else kind = 3;
            }
            // children onto the stack
            {
                int nch = kind == 3 ? nd.w : 0;
                int tot;
                int off = wave_excl_scan(nch, lane, tot);
                if (sp + tot > STACK_MAX) {
                    overflow = true;
                    break;
                }
#pragma unroll
                for (int c = 0; c < 8; c++)
                    if (c < nch) sset(sp + off + c, ((nd.z + c) << 5) | nb);
                sp += tot;
                wave_sync();
            }
            // accepted nodes
            {
                int tot;
                int off = wave_excl_count(kind == 1, tot);
                if (kind == 1) pcidx[pc_n + off] = e;
                pc_n += tot;
                wave_sync();
                if (pc_n >= 64) {
                    flush_pc(0, 64);
                    pc_n -= 64;
                    int t = (lane < pc_n) ? pcidx[64 + lane] : 0;
                    wave_sync();
                    if (lane < pc_n) pcidx[lane] = t;
                    wave_sync();
                }
            }
            // opened leaves: their particles
            {
                int rem = kind == 2 ? nd.y : 0;
                int pb = nd.x;
                for (;;) {
                    int tk = min(rem, PP_TAKE);
                    int tot;
                    int off = wave_excl_scan(tk, lane, tot);
                    if (tot == 0) break;
                    if (pp_n + tot > PP_CAP) {
                        int full = pp_n & ~63;
                        if (full) flush_pp(0, full / 64, 64);
                        int left = pp_n - full;
                        uint32_t t = (lane < left) ? ppidx[full + lane] : 0u;
                        wave_sync();
                        if (lane < left) ppidx[lane] = t;
                        wave_sync();
                        pp_n = left;
                    }
                    for (int t = 0; t < tk; t++) ppidx[pp_n + off + t] = ((uint32_t)(pb + t) << 5) | (uint32_t)nb;
                    pp_n += tot;
                    pb += tk;
                    rem -= tk;
                    wave_sync();
                }
                if (pp_n >= 64) {
                    int full = pp_n & ~63;
                    flush_pp(0, full / 64, 64);
                    int left = pp_n - full;
                    uint32_t t = (lane < left) ? ppidx[full + lane] : 0u;
                    wave_sync();
                    if (lane < left) ppidx[lane] = t;
                    wave_sync();
                    pp_n = left;
                }
            }
        }
        if (pc_n > 0) flush_pc(0, pc_n);
        if (pp_n > 0) flush_pp(0, 1, pp_n);
        if (fill > 0) {  // the last, partial chunk: far zero-mass dummies after the staged particles
            if (lane >= fill) cpp[lane] = to_src(dummy);
            wave_sync();
            pp_chunk();
            npp += (unsigned long long)fill;
            wave_sync();
        }
        // sum the R partial accumulators of each target (lanes tgt, tgt + Tw, ...)
        for (int o = Tw; o < 64; o <<= 1) {
#pragma unroll
            for (int i = 0; i < M; i++) {
                ax[i] += __shfl_xor(ax[i], o, 64);
                ay[i] += __shfl_xor(ay[i], o, 64);
                az[i] += __shfl_xor(az[i], o, 64);
            }
        }
        // The kick is written to its own arrays rather than added to the velocities, so the walk
        // can run while the PM kick of the same step updates them; the drift (or, for a tree
        // kick alone, an add kernel) adds it afterwards, in the same order as v += pm; v += tree.
        if (overflow && lane == 0) {
            atomicAdd(&A.counters[2], 1ull);
            atomicOr(&A.dsz[DSZ_WALKOVF], 1u);  // the step's drift reads it and leaves the box unmoved
        }
#pragma unroll
        for (int i = 0; i < M; i++) {
            if (valid[i] && rep == 0) {
                gst(A.tvx)[me[i]] = overflow ? 0.0 : (double)(A.fact * ax[i]);
                gst(A.tvy)[me[i]] = overflow ? 0.0 : (double)(A.fact * ay[i]);
                gst(A.tvz)[me[i]] = overflow ? 0.0 : (double)(A.fact * az[i]);
            }
        }
        if (lane == 0) {
            // (global atomics: a flat one would hold up the next group's first LDS wait)
            __hip_atomic_fetch_add(gst(A.counters), npp * (unsigned long long)cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(gst(A.counters) + 1, npc * (unsigned long long)cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if constexpr (CENSUS) {
            for (int o = 32; o > 0; o >>= 1) nin += (unsigned)__shfl_xor((int)nin, o, 64);
            if (lane == 0) __hip_atomic_fetch_add(gst(A.counters) + 3, (unsigned long long)nin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        };
        if (M == 3) group_body(ic<3>{});
        else group_body(ic<1>{});
    }
}

// FP64 walk: the same tree, groups and criteria in FP64 throughout, one wavefront per target group. (With
// one thread per target, depth first, 64 lanes read 64 nodes and leaves of their own from L2, and table
// lines too: theta = 0.5, 32^3 2.95 ms, 64^3 6.2, 128^3 26.3; this: 0.50, 1.37, 5.0.) A wave pops up to
// 64 nodes of its group's stack at a time, one per lane, and its targets share the accepted nodes and
// the listed sources. Sources are staged in LDS 64 at a time (those beyond the cutoff from the group's
// box dropped), the pair term's table lines (value and slope, 80 KB) are in LDS, and lane (slot, rep)
// sums every R-th source for its M targets. 16 waves and one table fill a CU's LDS. A team of 1 or 4
// waves takes a group: each wave walks down the same way until the stack holds enough nodes, then
// keeps every S-th of them (before that it takes every S-th of the accepted nodes and leaves), and the
// team's sums meet in LDS in a fixed order.
// What bounds it: FP64 issue in the pair loop (about 20 operations a pair) for large boxes, the
// heaviest group's own time for small ones.
struct walk64_args {
    const double *x, *y, *z;
    const int4* link;  // first particle, count, first child record, children
    const double* nd;
    const int* cellroot;
    const uint64_t* key;
    int cell_shift;
    const double* tab;
    int nbins;
    float lam;
    double *vx, *vy, *vz;
    unsigned long long* counters;
    const uint32_t* dsz;
    const int2* groups;
    uint32_t* ticket;
    int team;  // waves per group: 1 or 4
    int mcell;
    double box, rc2, rcut, inv_theta2, fact;
    int naccept;
    // sampled walk: group g is the particle groups[g].x alone (the per-particle test), its
    // acceleration written to out[3g..3g+2] (velocities untouched)
    double* out;
    uint32_t nsample;
};

constexpr int W64_STACK = 512;  // stack entries per wave; a pop takes no more nodes than leave room for their children
constexpr int W64_SLOTS = 2048;  // listed particles of one expansion (a bit each)

__device__ inline double wave_min64(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ inline double wave_max64(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

template <bool LOGT>
__global__ void __launch_bounds__(WALK_THREADS) walk_f64_kernel(walk64_args A) {
    __shared__ double2 s_tab[TAB_LDS];  // value and slope of the pair term
    __shared__ int s_stack[WALK_WAVES][W64_STACK];
    __shared__ double s_src[WALK_WAVES][3][64];
    __shared__ uint32_t s_head[WALK_WAVES][W64_SLOTS / 32];
    __shared__ int2 s_leaf[WALK_WAVES][64];
    __shared__ int s_pc[WALK_WAVES][64];
    __shared__ uint32_t s_bar[WALK_WAVES], s_next[WALK_WAVES];  // per team: arrivals, next group
    if (threadIdx.x < WALK_WAVES) s_bar[threadIdx.x] = 0u;
    for (int i = threadIdx.x; i < A.nbins; i += WALK_THREADS) s_tab[i] = make_double2(A.tab[6 * i], A.tab[6 * i + 1]);
    __syncthreads();
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int* stack = s_stack[wid];
    double *sx = s_src[wid][0], *sy = s_src[wid][1], *sz = s_src[wid][2];
    uint32_t* head = s_head[wid];
    int2* leaf = s_leaf[wid];
    int* pcl = s_pc[wid];
    const uint32_t ngroups = A.dsz[DSZ_OVERFLOW] ? 0u : (A.out ? A.nsample : A.dsz[DSZ_GROUPS]);
    const int S = A.team, team = wid / S, part = wid & (S - 1);
    const uint32_t nteams = gridDim.x * (uint32_t)(WALK_WAVES / S);
    uint32_t arrived = 0;
    // All waves of the team have written their LDS when it returns. Every wave of a team takes the
    // same groups and so as many of these waits as the others, and all are resident: each ends.
    auto team_sync = [&]() {
        wave_sync();
        if (S == 1) return;
        arrived += (uint32_t)S;
        if (lane == 0) {
            __hip_atomic_fetch_add(&s_bar[team], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
            while (__hip_atomic_load(&s_bar[team], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < arrived) __builtin_amdgcn_s_sleep(1);
        }
        wave_sync();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    const double rc2_keep = A.rc2 * (1.0 + 1e-12);  // a source beyond it from the group's box adds exactly zero
    unsigned long long npp = 0, npc = 0;
    // the first group by rank (the teams of one CU far apart: few groups spread over all CUs), the
    // others by ticket (see the FP32 walk)
    for (uint32_t g = (uint32_t)team * gridDim.x + blockIdx.x; g < ngroups;) {
        const int2 gr = A.groups[g];
        const int gbeg = __builtin_amdgcn_readfirstlane(gr.x), cnt = __builtin_amdgcn_readfirstlane(gr.y);
        // lanes (slot, rep): slots x R of them, M targets each; three targets a lane where that uses
        // at least as many lanes, and for groups of more than 64
        const int s3 = (cnt + 2) / 3, R3 = 64 / s3, R1 = cnt <= 64 ? 64 / cnt : 0;
        uint32_t next = 0u;
        auto group_body = [&](auto mc) {
            constexpr int M = decltype(mc)::value;
            const int slots = M == 3 ? s3 : cnt, R = M == 3 ? R3 : R1;
            const int rep = lane / slots, slot = lane - rep * slots;
            const bool act = rep < R;
            double xt[M], yt[M], zt[M], ax[M], ay[M], az[M];
            int me[M];
            bool valid[M];
            double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
#pragma unroll
            for (int i = 0; i < M; i++) {
                const int t = slot + i * slots;
                valid[i] = act && t < cnt;
                me[i] = gbeg + (valid[i] ? t : 0);  // an idle lane repeats target 0: inside the group's box
                xt[i] = A.x[me[i]]; yt[i] = A.y[me[i]]; zt[i] = A.z[me[i]];
                ax[i] = ay[i] = az[i] = 0.0;
                lo[0] = fmin(lo[0], xt[i]); hi[0] = fmax(hi[0], xt[i]);
                lo[1] = fmin(lo[1], yt[i]); hi[1] = fmax(hi[1], yt[i]);
                lo[2] = fmin(lo[2], zt[i]); hi[2] = fmax(hi[2], zt[i]);
            }
#pragma unroll
            for (int a = 0; a < 3; a++) {
                lo[a] = wave_min64(lo[a]);
                hi[a] = wave_max64(hi[a]);
            }
            // all group members share a chaining cell: the level-L prefix of their Morton key
            const uint64_t cellkey = A.key[gbeg] >> A.cell_shift;
            const int cx = (int)compact3(cellkey), cy = (int)compact3(cellkey >> 1), cz = (int)compact3(cellkey >> 2);
            auto shift_of = [&](int nb, double& qx, double& qy, double& qz) {
                const int tx = cx + nb % 3 - 1, ty = cy + (nb / 3) % 3 - 1, tz = cz + nb / 9 - 1;
                qx = tx < 0 ? -A.box : (tx >= A.mcell ? A.box : 0.0);
                qy = ty < 0 ? -A.box : (ty >= A.mcell ? A.box : 0.0);
                qz = tz < 0 ? -A.box : (tz >= A.mcell ? A.box : 0.0);
            };
            auto box_dist2 = [&](double qx, double qy, double qz) {
                const double ddx = fmax(fmax(lo[0] - qx, qx - hi[0]), 0.0);
                const double ddy = fmax(fmax(lo[1] - qy, qy - hi[1]), 0.0);
                const double ddz = fmax(fmax(lo[2] - qz, qz - hi[2]), 0.0);
                return ddx * ddx + ddy * ddy + ddz * ddz;
            };
            int sp = 0;
            {
                int e = -1;
                if (lane < 27) {
                    const int dx = lane % 3 - 1, dy = (lane / 3) % 3 - 1, dz = lane / 9 - 1;
                    const int nx = (cx + dx + A.mcell) % A.mcell, ny = (cy + dy + A.mcell) % A.mcell, nz = (cz + dz + A.mcell) % A.mcell;
                    const int r = A.cellroot[nx + A.mcell * (ny + A.mcell * nz)];
                    if (r >= 0) e = (r << 5) | lane;
                }
                const int off = wave_excl_count(e >= 0, sp);
                if (e >= 0) stack[off] = e;
                wave_sync();
            }
            bool split = S == 1;  // the stack holds this wave's share alone
            int fill = 0;  // staged sources, wave-uniform
            auto pp_chunk = [&](int m) {
                if (!act) return;
                for (int k = rep; k < m; k += R) {
                    const double qx = sx[k], qy = sy[k], qz = sz[k];
#pragma unroll
                    for (int i = 0; i < M; i++) {
                        const double dx = xt[i] - qx, dy = yt[i] - qy, dz = zt[i] - qz;
                        const double r2 = dx * dx + dy * dy + dz * dz;
                        double t;
                        const double2 tb = s_tab[table_bin64<LOGT>(r2, t, A.lam)];
                        const double f = r2 <= A.rc2 ? tb.x + tb.y * t : 0.0;  // unit particle mass
                        ax[i] += dx * f; ay[i] += dy * f; az[i] += dz * f;
                    }
                }
            };
            // particles of 64 slots (in: this lane's slot holds one), those near the group to the chunk
            auto stage = [&](bool in, int p, int nb) {
                double qx = 0.0, qy = 0.0, qz = 0.0;
                if (in) {
                    double hx, hy, hz;
                    shift_of(nb, hx, hy, hz);
                    qx = A.x[p] + hx; qy = A.y[p] + hy; qz = A.z[p] + hz;
                }
                const bool keep = in && box_dist2(qx, qy, qz) <= rc2_keep;
                int tot;
                const int off = wave_excl_count(keep, tot);
                const int room = 64 - fill;
                if (keep && off < room) { sx[fill + off] = qx; sy[fill + off] = qy; sz[fill + off] = qz; }
                fill += tot;
                wave_sync();
                if (fill >= 64) {
                    pp_chunk(64);
                    wave_sync();
                    if (keep && off >= room) { sx[off - room] = qx; sy[off - room] = qy; sz[off - room] = qz; }
                    fill -= 64;
                    wave_sync();
                }
            };
            // the particles of the lanes' leaves (first particle, count; count 0: none): slot s of an
            // expansion belongs to the last leaf whose first slot is not after it, found by counting
            // the marks of first slots
            auto leaves = [&](int first, int count, int nb) {
                for (int done = 0; done < 64;) {
                    int all;
                    const int c = lane >= done ? min(count, W64_SLOTS + 1) : 0;
                    const int P = wave_excl_scan(c, lane, all);
                    if (all == 0) break;
                    // lanes done .. m - 1 fit (a prefix); none: lane `done` alone holds more than the marks cover
                    const int m = __builtin_amdgcn_readfirstlane(__popcll(__ballot(P + c <= W64_SLOTS)));
                    if (m <= done) {
                        const int b0 = __builtin_amdgcn_readlane(first, done), n0 = __builtin_amdgcn_readlane(count, done);
                        const int nb0 = __builtin_amdgcn_readlane(nb, done);
                        npp += (unsigned long long)n0 * (unsigned)cnt;
                        for (int s = 0; s < n0; s += 64) stage(s + lane < n0, b0 + s + lane, nb0);
                        done++;
                        continue;
                    }
                    const int T = __builtin_amdgcn_readlane(P + c, m - 1);
                    npp += (unsigned long long)T * (unsigned)cnt;
                    if (32 * lane < T) head[lane] = 0u;
                    wave_sync();
                    int held;
                    const bool has = lane >= done && lane < m && c > 0;
                    const int k = wave_excl_count(has, held);
                    if (has) {
                        atomicOr(&head[P >> 5], 1u << (P & 31));
                        leaf[k] = make_int2(first - P, nb);
                    }
                    wave_sync();
                    int before = -1;
                    for (int s0 = 0; s0 < T; s0 += 64) {
                        const unsigned wl = (unsigned)__builtin_amdgcn_readfirstlane((int)head[s0 >> 5]);
                        const unsigned wh = (unsigned)__builtin_amdgcn_readfirstlane((int)head[(s0 >> 5) + 1]);
                        const unsigned long long w = ((unsigned long long)wh << 32) | wl, w1 = w >> 1;
                        const int j = before + (int)(wl & 1u) +
                                      (int)__builtin_amdgcn_mbcnt_hi((unsigned)(w1 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)w1, 0u));
                        before += __popcll(w);
                        const bool in = s0 + lane < T;
                        const int2 e = leaf[in ? j : 0];
                        stage(in, e.x + s0 + lane, e.y);
                    }
                    done = m;
                }
            };
            while (sp > 0) {
                // after a pop of `take` nodes at most 7 take more entries: kept below the stack's end
                // less 128; a single node at a time always fits (7 more entries a level, 14 levels)
                const int take = min(min(sp, 64), max(1, (W64_STACK - 128 - sp) / 7));
                sp -= take;
                const int e = lane < take ? stack[sp + lane] : -1;
                wave_sync();
                int kind = 0;  // 0 none, 1 accept, 2 leaf, 3 open
                int4 nd = make_int4(0, 0, 0, 0);
                int v = 0, nb = 0;
                if (e >= 0) {
                    v = e >> 5;
                    nb = e & 31;
                    double hx, hy, hz;
                    shift_of(nb, hx, hy, hz);
                    const double* m = A.nd + 12 * (size_t)v;
                    nd = A.link[v];
                    const double rmax = m[11];
                    const double dmin2 = box_dist2(m[0] + hx, m[1] + hy, m[2] + hz);
                    const double rr = A.rcut + rmax;
                    if (dmin2 > rr * rr) kind = 0;
                    else if (nd.y >= A.naccept && dmin2 >= rmax * rmax * A.inv_theta2) kind = 1;
                    else kind = nd.w == 0 ? 2 : 3;
                }
                int tot;
                const int nch = kind == 3 ? nd.w : 0;
                const int off = wave_excl_scan(nch, lane, tot);
                for (int c = 0; c < nch; c++) stack[sp + off + c] = ((nd.z + c) << 5) | nb;
                sp += tot;
                wave_sync();
                if (!split && (lane & (S - 1)) != part) kind = 0;  // another wave's
                if (!split && sp >= 16 * S) {
                    const int n = (sp - part + S - 1) / S;
                    for (int k = 0; k < n; k += 64) {  // (entries move towards the bottom: read, then written)
                        const int q = k + lane < n ? stack[(k + lane) * S + part] : 0;
                        wave_sync();
                        if (k + lane < n) stack[k + lane] = q;
                        wave_sync();
                    }
                    sp = n;
                    split = true;
                }
                int nacc;
                const int poff = wave_excl_count(kind == 1, nacc);
                if (kind == 1) pcl[poff] = e;
                wave_sync();
                npc += (unsigned long long)nacc * (unsigned)cnt;
                if (act) {
                    for (int k = rep; k < nacc; k += R) {
                        const int q = pcl[k];
                        double hx, hy, hz;
                        shift_of(q & 31, hx, hy, hz);
                        const double* m = A.nd + 12 * (size_t)(q >> 5);
                        const double qx = m[0] + hx, qy = m[1] + hy, qz = m[2] + hz;
#pragma unroll
                        for (int i = 0; i < M; i++) {
                            const double dx = xt[i] - qx, dy = yt[i] - qy, dz = zt[i] - qz;
                            const double r2 = dx * dx + dy * dy + dz * dz;
                            if (r2 > A.rc2) continue;
                            double t;
                            const double* tb = A.tab + 6 * table_bin64<LOGT>(r2, t, A.lam);
                            const double f1 = tb[0] + tb[1] * t, f2 = tb[2] + tb[3] * t, f3 = tb[4] + tb[5] * t;
                            const double qx1 = m[4] * dx + m[7] * dy + m[8] * dz;
                            const double qx2 = m[7] * dx + m[5] * dy + m[9] * dz;
                            const double qx3 = m[8] * dx + m[9] * dy + m[6] * dz;
                            const double qxy = dx * qx1 + dy * qx2 + dz * qx3;
                            const double tmp = m[3] * f1 + m[10] * f2 + qxy * f3;
                            ax[i] += dx * tmp + qx1 * 2 * f2;
                            ay[i] += dy * tmp + qx2 * 2 * f2;
                            az[i] += dz * tmp + qx3 * 2 * f2;
                        }
                    }
                }
                leaves(nd.x, kind == 2 ? nd.y : 0, nb);
            }
            if (fill > 0) pp_chunk(fill);
            wave_sync();
            // the R partial sums of each target in each of the team's waves, in a fixed order (the
            // chunk's LDS is free now); the team's first wave adds them up and takes the next group
            if (part == 0 && lane == 0) s_next[team] = nteams + atomicAdd(A.ticket, 1u);
#pragma unroll
            for (int i = 0; i < M; i++) {
                sx[lane] = ax[i]; sy[lane] = ay[i]; sz[lane] = az[i];
                team_sync();
                // The next group is read between the last two waits: the first wave writes the one after
                // it only past the second of them, when every wave of the team has read this one.
                if (i == M - 1) next = *(volatile uint32_t*)&s_next[team];
                if (part == 0 && rep == 0 && valid[i]) {
                    double fx = 0.0, fy = 0.0, fz = 0.0;
                    for (int w = 0; w < S; w++)
                        for (int r = 0; r < R; r++) {
                            fx += s_src[wid + w][0][slot + r * slots];
                            fy += s_src[wid + w][1][slot + r * slots];
                            fz += s_src[wid + w][2][slot + r * slots];
                        }
                    if (A.out) {
                        A.out[3 * (size_t)g] = A.fact * fx;
                        A.out[3 * (size_t)g + 1] = A.fact * fy;
                        A.out[3 * (size_t)g + 2] = A.fact * fz;
                    } else {
                        A.vx[me[i]] += A.fact * fx;
                        A.vy[me[i]] += A.fact * fy;
                        A.vz[me[i]] += A.fact * fz;
                    }
                }
                team_sync();
            }
        };
        if (R3 >= 3 * R1) group_body(ic<3>{});
        else group_body(ic<1>{});
        g = (uint32_t)__builtin_amdgcn_readfirstlane((int)next);
    }
    if (lane == 0 && (npp | npc)) {
        atomicAdd(&A.counters[0], npp);
        atomicAdd(&A.counters[1], npc);
    }
}

unsigned blocks_for(size_t n, int t) { return (unsigned)std::max<size_t>(1, (n + t - 1) / t); }

template <typename T>
int regrow(lagpm_ctx* ctx, T** p, size_t count) {
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    HIPCHK(ctx, hipMalloc((void**)p, std::max<size_t>(count, 1) * sizeof(T)));
    return LAGPM_OK;
}

}  // namespace

int lagpm_choose_cell_level(int n, double rsphere) {
    int L = 0;
    while (L < LAGPM_KEY_BITS && (double)n / (double)(1 << (L + 1)) >= rsphere) L++;
    return L;
}

size_t lagpm_tree_node_cap_guess(size_t np, int mcell) {
    // nleaf = 16 gives about np/6 nodes for uniform and np/4 for strongly clustered input
    return np / 3 + (size_t)mcell * mcell * mcell + 4096;
}

// scale of the FP32 tree's coordinates: sqrt(lam) for the log-r^2 tables, 1 for the r-table law
double lagpm_tree_scale(const lagpm_box* box) {
    return box->tab && box->tab->logr2 ? std::sqrt((double)box->tab->lam) : 1.0;
}

// scratch of a build: counts and offsets of the particle blocks' rows and of the node blocks' groups
static size_t tree_part_blocks(size_t np) { return (np + TB_PART - 1) / TB_PART; }
static size_t tree_group_blocks(size_t cap) { return (cap + GB_NODES - 1) / GB_NODES; }
size_t lagpm_tree_tmp_bytes(size_t np, size_t cap) {
    return 2 * (TB_ROWS * tree_part_blocks(np) + tree_group_blocks(cap)) * sizeof(uint32_t);
}

int lagpm_tree_alloc(lagpm_ctx* ctx, lagpm_box* box, size_t cap) {
    const bool f64 = box->p.precision == LAGPM_PREC_FP64;
    if (cap > (size_t)LAGPM_MAX_NODES) {
        if (box->node_cap >= (size_t)LAGPM_MAX_NODES)
            return lagpm_fail(ctx, LAGPM_E_INVAL, "tree needs more than 2^26 nodes (the walk's node index limit)");
        cap = LAGPM_MAX_NODES;
    }
    const size_t gcap = cap + box->np / 64 + 1;
    box->node_cap = box->group_cap = 0;  // none until all are there: the old arrays go first
    RCHK(regrow(ctx, &box->nd_link, cap));
    RCHK(regrow(ctx, &box->nd_lev, cap));
    RCHK(regrow(ctx, &box->nd_rop, cap));
    RCHK(regrow(ctx, &box->groups, gcap));
    if (f64) {
        RCHK(regrow(ctx, &box->nd_d, 12 * cap));
    } else {
        RCHK(regrow(ctx, &box->nd_geo, cap));
        RCHK(regrow(ctx, &box->nd_q0, cap));
        RCHK(regrow(ctx, &box->nd_q1, cap));
    }
    const size_t need = std::max(lagpm_tree_tmp_bytes(box->np, cap), lagpm_sort_tmp_bytes(box->np));
    if (need > box->scan_tmp_bytes) {  // (small; sorts go on with the old one if this fails)
        uint32_t* tmp = nullptr;
        RCHK(regrow(ctx, (char**)&tmp, need));
        if (box->scan_tmp) (void)hipFree(box->scan_tmp);
        box->scan_tmp = tmp;
        box->scan_tmp_bytes = need;
    }
    box->node_cap = cap;
    box->group_cap = gcap;
    return LAGPM_OK;
}

// The tree is expected to end above box->depth, so only the top 3 * depth key bits must be in order:
// a box whose tree is shallower needs fewer passes. Below them the order is the previous one (the
// sort is stable). An even number of passes leaves the result in key/perm, where the gather and the
// walk's descriptors expect it.
static int sort_passes(const lagpm_box* box) {
    const int D = std::min(LAGPM_KEY_BITS, std::max(box->level_cell, box->depth));
    return (((3 * D + 7) / 8) + 1) & ~1;
}
// Levels a build may split to: down to box->depth, and a tree that needs more is detected and
// redone after a full sort; but where the passes have put all key bits in order (depth 11 and more)
// the build goes on below the limit itself, and gives what the redone one would. A halo that
// tightens costs no second sort, build and walk then: a batch of 10 boxes (32^3-96^3) redid 9 trees in
// 10 steps and took 5 of its 53 ms over them. The levels below the limit take their moments in one
// launch: a launch each cost a 64^3 step 0.02 of 1.01 ms.
static int build_depth(const lagpm_box* box) {
    if (8 * sort_passes(box) >= 3 * LAGPM_KEY_BITS) return LAGPM_KEY_BITS;
    return std::min(LAGPM_KEY_BITS, std::max(box->level_cell, box->depth));
}

int lagpm_sort_bits(const lagpm_box* box) { return 8 * sort_passes(box); }

int lagpm_sort_particles(lagpm_ctx* ctx, lagpm_box* box, const double* drag, hipStream_t vst) {
    const size_t np = box->np;
    if (np == 0) return LAGPM_OK;
    hipStream_t st = box->st;
    const double s = 65536.0 / (double)box->p.n;
    hipLaunchKernelGGL(keys_kernel, dim3(blocks_for(np, 256)), dim3(256), 0, st, box->x, box->y, box->z, np, s,
                       box->key, box->perm);
    HIPCHK(ctx, hipGetLastError());
    const int passes = sort_passes(box);
    bool alt = false;
    RCHK(lagpm_radix_sort_pairs(ctx, st, box->scan_tmp, box->key, box->key2, box->perm, box->perm2, np, 8 * passes, &alt,
                                3 * LAGPM_KEY_BITS - 8 * passes));
    if (alt) return lagpm_fail(ctx, LAGPM_E_STATE, "radix sort ended in the scratch buffers");
    double** arrs[6] = {&box->x, &box->y, &box->z, &box->vx, &box->vy, &box->vz};
    gather_set g;
    for (int a = 0; a < 6; a++) {
        g.src[a] = *arrs[a];
        g.dst[a] = box->alt[a];
    }
    g.id = box->id;
    g.id_dst = box->id_alt;
    if (vst && vst != st) {
        // the positions first, alone (everything after the sort waits for them), then the
        // velocities and ids on vst beside what follows; the caller joins box->evvel before using them
        hipLaunchKernelGGL(gather_pos_kernel, dim3(blocks_for(np, 256)), dim3(256), 0, st, g, box->perm, np);
        HIPCHK(ctx, hipGetLastError());
        HIPCHK(ctx, hipEventRecord(box->evsort, st));
        HIPCHK(ctx, hipStreamWaitEvent(vst, box->evsort, 0));
        hipLaunchKernelGGL(gather_vel_kernel, dim3(blocks_for(np, 256)), dim3(256), 0, vst, g, box->perm, np, drag);
        HIPCHK(ctx, hipGetLastError());
        HIPCHK(ctx, hipEventRecord(box->evvel, vst));
    } else {
        hipLaunchKernelGGL(gather_all_kernel, dim3(blocks_for(np, 256)), dim3(256), 0, st, g, box->perm, np, drag);
    }
    HIPCHK(ctx, hipGetLastError());
    for (int a = 0; a < 6; a++) std::swap(*arrs[a], box->alt[a]);
    std::swap(box->id, box->id_alt);
    box->sorted = true;
    box->sorted_bits = 8 * passes;
    return LAGPM_OK;
}

int lagpm_tree_build(lagpm_ctx* ctx, lagpm_box* box) {
    const size_t np = box->np;
    const int L = box->level_cell;
    const int nleaf = box->tune.nleaf;
    const int G = box->tune.group;
    const bool f64 = box->p.precision == LAGPM_PREC_FP64;
    hipStream_t st = box->st;
    // an earlier growth of the node arrays failed and left none
    if (box->node_cap == 0) RCHK(lagpm_tree_alloc(ctx, box, lagpm_tree_node_cap_guess(np, box->mcell)));
    const size_t cap = box->node_cap, gcap = box->group_cap;
    if (np == 0) {
        hipLaunchKernelGGL(tree_reset_kernel, dim3(1), dim3(64), 0, st, box->dsz, box->counters);
        HIPCHK(ctx, hipGetLastError());
        return LAGPM_OK;
    }
    // (the depth limit may have been raised since the last sort: lagpm_box_set_tuning)
    if (!lagpm_sorted_for_build(box)) RCHK(lagpm_sort_particles(ctx, box));
    const size_t ncell = (size_t)box->mcell * box->mcell * box->mcell;
    const int D = build_depth(box);
    const uint32_t nblk = (uint32_t)tree_part_blocks(np), gblk = (uint32_t)tree_group_blocks(cap);
    uint32_t* cnt = box->scan_tmp;
    uint32_t* off = cnt + (size_t)TB_ROWS * nblk;
    uint32_t* gcnt = off + (size_t)TB_ROWS * nblk;
    uint32_t* goff = gcnt + gblk;
    hipLaunchKernelGGL(tree_count_kernel, dim3(std::max(nblk, blocks_for(ncell, 4 * TB_THREADS))), dim3(TB_THREADS), 0, st, box->key,
                       np, nleaf, L, D, box->x, box->y, box->z, f64 ? 1.0 : lagpm_tree_scale(box), f64 ? (float4*)nullptr : box->pp,
                       box->cellroot, ncell, cnt, nblk);
    HIPCHK(ctx, hipGetLastError());
    hipLaunchKernelGGL(tree_rows_kernel, dim3((unsigned)(D - L + 3)), dim3(256), 0, st, cnt, off, nblk, L, D, box->dsz, box->counters);
    HIPCHK(ctx, hipGetLastError());
    hipLaunchKernelGGL(tree_emit_kernel, dim3(nblk), dim3(TB_THREADS), 0, st, box->key, np, nleaf, L, D, off, nblk, cap, box->dsz,
                       box->nd_link, box->nd_lev, box->nd_rop, box->cellroot, box->mcell);
    HIPCHK(ctx, hipGetLastError());
    const unsigned mblocks = (unsigned)std::min<size_t>(2 * LEVEL_BLOCKS, blocks_for(cap * MOM_ROW, 256));
    const int expected = std::min(D, std::max(L, box->depth));
    if (expected < D) {
        if (f64)
            hipLaunchKernelGGL(moments_f64_deep_kernel, dim3(1), dim3(MOM_DEEP_THREADS), 0, st, box->x, box->y, box->z, box->dsz, D,
                               expected + 1, box->nd_lev, box->nd_link, box->nd_d);
        else
            hipLaunchKernelGGL(moments_f32_deep_kernel, dim3(1), dim3(MOM_DEEP_THREADS), 0, st, box->pp, box->dsz, D, expected + 1,
                               box->nd_lev, box->nd_link, box->nd_geo, box->nd_q0, box->nd_q1);
        HIPCHK(ctx, hipGetLastError());
    }
    for (int l = expected; l >= L; l--) {  // levels below D hold no records
        if (f64)
            hipLaunchKernelGGL(moments_f64_kernel, dim3(mblocks), dim3(256), 0, st, box->x, box->y, box->z, box->dsz, l, box->nd_lev,
                               box->nd_link, box->nd_d);
        else
            hipLaunchKernelGGL(moments_f32_kernel, dim3(mblocks), dim3(256), 0, st, box->pp, box->dsz, l, box->nd_lev, box->nd_link,
                               box->nd_geo, box->nd_q0, box->nd_q1);
        HIPCHK(ctx, hipGetLastError());
    }
    const int runs = box->tune.runs;
    hipLaunchKernelGGL(group_count_kernel, dim3(gblk), dim3(GB_THREADS), 0, st, box->dsz, cap, L, G, runs, box->nd_link, box->nd_lev,
                       box->nd_rop, gcnt);
    HIPCHK(ctx, hipGetLastError());
    hipLaunchKernelGGL(group_rows_kernel, dim3(1), dim3(256), 0, st, gcnt, goff, gblk, gcap, box->dsz);
    HIPCHK(ctx, hipGetLastError());
    hipLaunchKernelGGL(group_write_kernel, dim3(gblk), dim3(GB_THREADS), 0, st, box->dsz, cap, L, G, runs, box->nd_link, box->nd_lev,
                       box->nd_rop, goff, box->groups);
    HIPCHK(ctx, hipGetLastError());
    box->tree_built = true;
    return LAGPM_OK;
}

int lagpm_tree_walk_f32(lagpm_ctx* ctx, lagpm_box* const* boxes, const double* facts, int nbox, int reserve_cu,
                        const walk_sample* sample) {
    if (nbox <= 0) return LAGPM_OK;
    if (sample && nbox != 1) return lagpm_fail(ctx, LAGPM_E_INVAL, "a sampled walk takes one box");
    if ((size_t)nbox > ctx->walk_box_cap) {
        size_t cap = std::max<size_t>(64, (size_t)nbox * 2);
        ctx->walk_box_cap = 0;
        RCHK(regrow(ctx, &ctx->walk_boxes, cap));
        RCHK(regrow(ctx, &ctx->walk_prefix, cap + 1));
        ctx->walk_box_cap = cap;
    }
    const law_tables* tab = boxes[0]->tab;
    std::vector<walk_box> hb((size_t)nbox);
    for (int b = 0; b < nbox; b++) {
        lagpm_box* box = boxes[b];
        if (box->tab != tab || box->p.precision != LAGPM_PREC_FP32)
            return lagpm_fail(ctx, LAGPM_E_INVAL, "boxes of one walk launch must share the FP32 force table");
        const double th = box->p.theta;
        walk_box& A = hb[(size_t)b];
        A.pp = box->pp; A.link = box->nd_link; A.geo = box->nd_geo; A.q0 = box->nd_q0;
        A.q1 = box->nd_q1; A.cellroot = box->cellroot; A.groups = box->groups; A.key = box->key;
        A.tvx = box->alt[0]; A.tvy = box->alt[1]; A.tvz = box->alt[2];  // free between sorts
        A.counters = box->counters; A.dsz = box->dsz;
        if (sample) {  // the sampled particles as groups of one (sizes: the sample's own words)
            A.groups = sample->groups;
            A.dsz = sample->dsz;
        }
        A.cell_shift = 3 * (LAGPM_KEY_BITS - box->level_cell);
        A.mcell = box->mcell;
        A.naccept = LAGPM_NACCEPT;
        // lengths in the units of pp (scaled by sc, see tree_count_kernel)
        const double sc = lagpm_tree_scale(box);
        A.box = (float)(box->p.n * sc);
        A.rc2 = (float)(box->p.rsphere * box->p.rsphere * sc * sc);
        A.rcut = (float)(box->p.rsphere * sc);
        A.inv_theta2 = (float)(th > 0 ? 1.0 / (th * th) : 1e30);
        A.fact = (float)(facts[b] * box->p.mass / ((double)box->p.n * (double)box->p.n) / sc);
    }
    // pageable source: the copy is staged before the call returns, so hb may go out of scope
    HIPCHK(ctx, hipMemcpyAsync(ctx->walk_boxes, hb.data(), hb.size() * sizeof(walk_box), hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(walk_prefix_kernel, dim3(1), dim3(64), 0, ctx->stream, ctx->walk_boxes, nbox, ctx->walk_prefix,
                       ctx->walk_ticket);
    HIPCHK(ctx, hipGetLastError());
    // each box's walk-start event, right before the launch (after the descriptor copy and the
    // prefix, so the phase time is the walk kernel's own)
    for (int b = 0; b < nbox; b++) HIPCHK(ctx, hipEventRecord(boxes[b]->ev[14], ctx->stream));
    // one workgroup per CU fills it (registers and LDS); reserve_cu CUs are left free for other
    // streams' kernels, in whole XCD rounds so every XCD keeps the same number of walk workgroups
    const int full = (int)(ctx->walk_stack_entries / ((size_t)STACK_MAX * WALK_WAVES));
    const int keep = full - ((std::max(0, reserve_cu) + WALK_XCDS - 1) / WALK_XCDS) * WALK_XCDS;
    const unsigned blocks = (unsigned)(keep >= WALK_XCDS ? keep : std::min(full, WALK_XCDS));
    auto kern = tab->logr2 ? (ctx->walk_census ? walk_f32_kernel<true, true> : walk_f32_kernel<true, false>)
                           : (ctx->walk_census ? walk_f32_kernel<false, true> : walk_f32_kernel<false, false>);
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(WALK_THREADS), 0, ctx->stream, ctx->walk_boxes, ctx->walk_prefix, nbox,
                       tab->tab0, tab->tab12, ctx->walk_stack, ctx->walk_ticket);
    HIPCHK(ctx, hipGetLastError());
    return LAGPM_OK;
}

int lagpm_tree_walk_f64(lagpm_ctx* ctx, lagpm_box* box, double fact, const walk_sample* sample) {
    if (box->np == 0) return LAGPM_OK;
    const double th = box->p.theta;
    walk64_args A;
    A.x = box->x; A.y = box->y; A.z = box->z; A.link = box->nd_link;
    A.nd = box->nd_d; A.cellroot = box->cellroot;
    A.key = box->key; A.cell_shift = 3 * (LAGPM_KEY_BITS - box->level_cell);
    A.tab = box->tab->tabd; A.nbins = box->tab->nbins; A.lam = box->tab->lam;
    A.vx = box->vx; A.vy = box->vy; A.vz = box->vz; A.counters = box->counters; A.dsz = box->dsz;
    A.groups = sample ? sample->groups : box->groups;
    A.ticket = (sample ? sample->dsz : box->dsz) + DSZ_TICKET;
    A.mcell = box->mcell; A.box = (double)box->p.n; A.rc2 = box->tab->rc2_eff;
    A.rcut = box->p.rsphere; A.inv_theta2 = th > 0 ? 1.0 / (th * th) : 1e30;
    A.fact = fact * box->p.mass / ((double)box->p.n * (double)box->p.n);
    A.naccept = LAGPM_NACCEPT;
    A.out = sample ? sample->out : nullptr;
    A.nsample = sample ? (uint32_t)sample->count : 0u;
    // Teams of four while a CU's waves get about two groups or less each: then the heaviest group's
    // own time is the walk's. Walk in ms with one wave and with four: 32^3 0.56 and 0.50, 64^3 1.81 and
    // 1.37, 72^3 (373,248 targets) 1.27 and 1.59, 96^3 2.3 and 3.0 (four waves each walk down to the split).
    const size_t targets = sample ? 44 * sample->count : box->np;
    A.team = targets <= 300000 ? 4 : 1;
    const unsigned blocks = (unsigned)std::max(1, ctx->num_cu);  // one workgroup per CU (its LDS)
    auto kern = box->tab->logr2 ? walk_f64_kernel<true> : walk_f64_kernel<false>;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(WALK_THREADS), 0, box->st, A);
    HIPCHK(ctx, hipGetLastError());
    return LAGPM_OK;
}

int lagpm_tree_readback_enqueue(lagpm_ctx* ctx, lagpm_box* box, tree_readback* dst) {
    HIPCHK(ctx, hipMemcpyAsync(dst->d, box->dsz, sizeof(dst->d), hipMemcpyDeviceToHost, box->st));
    HIPCHK(ctx, hipMemcpyAsync(dst->c, box->counters, sizeof(dst->c), hipMemcpyDeviceToHost, box->st));
    return LAGPM_OK;
}

int lagpm_tree_finish(lagpm_ctx* ctx, lagpm_box* box, bool* retry) {
    *retry = false;
    if (!ctx->readback1) HIPCHK(ctx, hipHostMalloc(&ctx->readback1, sizeof(tree_readback), hipHostMallocDefault));
    tree_readback* r = static_cast<tree_readback*>(ctx->readback1);
    RCHK(lagpm_tree_readback_enqueue(ctx, box, r));
    HIPCHK(ctx, hipStreamSynchronize(box->st));
    return lagpm_tree_finish_with(ctx, box, *r, retry);
}

int lagpm_tree_finish_with(lagpm_ctx* ctx, lagpm_box* box, const tree_readback& r, bool* retry) {
    *retry = false;
    const uint32_t* d = r.d;
    const unsigned long long* c = r.c;
    box->stats.n_pp = c[0];
    box->stats.n_pc = c[1];
    box->stats.n_pp_within = c[3];
    box->stats.n_nodes = d[DSZ_NODES];
    box->stats.n_groups = d[DSZ_GROUPS];
    if (d[DSZ_DEEPER]) {
        // the tree needs levels below the depth limit: redo it at full depth, with room for the
        // nodes the truncated build could not count
        box->depth = LAGPM_KEY_BITS;
        box->sorted = false;  // the keys are in order down to the old limit only: sort again
        const size_t need = std::max<size_t>((size_t)d[DSZ_NODES], box->node_cap);
        if (d[DSZ_NODES] >= box->node_cap) RCHK(lagpm_tree_alloc(ctx, box, need + need / 2 + 4096));
        *retry = true;
        return LAGPM_E_OVERFLOW;
    }
    if (d[DSZ_OVERFLOW]) {
        // grow to the node count this input needs (groups follow from nodes) and rebuild
        size_t need = std::max<size_t>((size_t)d[DSZ_NODES], box->node_cap);
        RCHK(lagpm_tree_alloc(ctx, box, need + need / 4 + 4096));
        *retry = true;
        return LAGPM_E_OVERFLOW;
    }
    int deepest = box->level_cell;
    for (int l = box->level_cell; l <= LAGPM_KEY_BITS; l++)
        if (d[DSZ_LVL + l]) deepest = l;
    box->stats.deepest = deepest;
    if (box->depth >= LAGPM_KEY_BITS) {
        // first complete build at full depth: limit later builds to two levels below its deepest
        box->depth = std::min(LAGPM_KEY_BITS, deepest + 2);
    } else if (deepest > box->depth) {  // a build below the limit (build_depth): as a rebuild would set it
        box->depth = std::min(LAGPM_KEY_BITS, deepest + 2);
    }
    if (c[2]) return lagpm_fail(ctx, LAGPM_E_OVERFLOW, "tree walk stack overflow in " + std::to_string(c[2]) + " groups");
    return LAGPM_OK;
}

namespace {
// slot[ids[t]] = t: the sample index of each sampled caller index (slot starts at -1)
__global__ void sample_slot_kernel(const int64_t* __restrict__ ids, size_t count, int* __restrict__ slot) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < count) slot[ids[t]] = (int)t;
}
__global__ void fill_i32_kernel(int* __restrict__ a, size_t m, int v) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (size_t)gridDim.x * blockDim.x) a[i] = v;
}
// every sample group starts as particle 0 alone (a valid group of one), then gets its particle
__global__ void sample_init_kernel(int2* __restrict__ groups, size_t count) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < count) groups[t] = make_int2(0, 1);
}
// sample t is the particle now at position p (the box's current order): a group of one at p
__global__ void sample_groups_kernel(const uint32_t* __restrict__ id, size_t np, const int* __restrict__ slot,
                                     int2* __restrict__ groups) {
    const size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const int t = slot[id[p]];
    if (t >= 0) groups[t] = make_int2((int)p, 1);
}
// the sample's size words: the box's (its overflow flag) with the group count replaced
__global__ void sample_dsz_kernel(const uint32_t* __restrict__ dsz, uint32_t* __restrict__ sdsz, uint32_t count) {
    for (int i = threadIdx.x; i < DSZ_COUNT; i += blockDim.x) sdsz[i] = i == DSZ_GROUPS ? count : (i == DSZ_TICKET ? 0u : dsz[i]);
}
__global__ void sample_gather_kernel(const int2* __restrict__ groups, size_t count, const double* __restrict__ tx,
                                     const double* __restrict__ ty, const double* __restrict__ tz, double* __restrict__ out) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    const int p = groups[t].x;
    out[3 * t] = tx[p];
    out[3 * t + 1] = ty[p];
    out[3 * t + 2] = tz[p];
}
}  // namespace

// Walks the sampled particles of a built tree, each alone; acc (device, 3 per sample) gets their
// accelerations. ids (device) are caller indices, distinct and below np (checked by the caller).
int lagpm_tree_walk_sample(lagpm_ctx* ctx, lagpm_box* box, const int64_t* ids, size_t count, int* slot, int2* groups,
                           uint32_t* sdsz, double* acc) {
    const size_t np = box->np;
    hipStream_t st = box->st;
    hipLaunchKernelGGL(fill_i32_kernel, dim3(blocks_for(np, 256)), dim3(256), 0, st, slot, np, -1);
    hipLaunchKernelGGL(sample_slot_kernel, dim3(blocks_for(count, 256)), dim3(256), 0, st, ids, count, slot);
    hipLaunchKernelGGL(sample_init_kernel, dim3(blocks_for(count, 256)), dim3(256), 0, st, groups, count);
    hipLaunchKernelGGL(sample_groups_kernel, dim3(blocks_for(np, 256)), dim3(256), 0, st, box->id, np, slot, groups);
    hipLaunchKernelGGL(sample_dsz_kernel, dim3(1), dim3(64), 0, st, box->dsz, sdsz, (uint32_t)count);
    HIPCHK(ctx, hipGetLastError());
    walk_sample smp{groups, sdsz, acc, count};
    if (box->p.precision == LAGPM_PREC_FP64) {
        RCHK(lagpm_tree_walk_f64(ctx, box, 1.0, &smp));
    } else {
        // the walk runs on the context stream and writes its kicks at the particles' positions
        if (st != ctx->stream) {
            HIPCHK(ctx, hipEventRecord(box->ev[10], st));
            HIPCHK(ctx, hipStreamWaitEvent(ctx->stream, box->ev[10], 0));
        }
        const double one = 1.0;
        RCHK(lagpm_tree_walk_f32(ctx, &box, &one, 1, 0, &smp));
        hipLaunchKernelGGL(sample_gather_kernel, dim3(blocks_for(count, 256)), dim3(256), 0, ctx->stream, groups, count,
                           (const double*)box->alt[0], (const double*)box->alt[1], (const double*)box->alt[2], acc);
        HIPCHK(ctx, hipGetLastError());
        if (st != ctx->stream) {
            HIPCHK(ctx, hipEventRecord(box->ev[11], ctx->stream));
            HIPCHK(ctx, hipStreamWaitEvent(st, box->ev[11], 0));
        }
    }
    return LAGPM_OK;
}

size_t lagpm_walk_stack_entries(int num_cu) {
    size_t blocks = (size_t)std::max(1, num_cu);  // one 16-wave workgroup per CU
    return blocks * WALK_WAVES * STACK_MAX;
}

// The octree of the last build in the box's own units: FP32 trees keep positions scaled by the
// tree scale s (see tree_count_kernel) and masses in particle masses; the FP64 tree keeps cells.
extern "C" int lagpm_tree_nodes_get(lagpm_ctx* ctx, lagpm_box* box, size_t cap, size_t* nnodes, int32_t* info,
                                    double* com, double* quad, uint32_t* order) {
    if (!ctx || !box || !nnodes) return lagpm_fail(ctx, LAGPM_E_INVAL, "NULL argument");
    *nnodes = 0;
    if (box->np == 0) return LAGPM_OK;
    if (!box->tree_built) return lagpm_fail(ctx, LAGPM_E_STATE, "no tree built: call lagpm_treecorrection first");
    HIPCHK(ctx, hipSetDevice(ctx->device));
    uint32_t d[DSZ_COUNT];
    RCHK(lagpm_d2h(ctx, d, box->dsz, sizeof(d), box->st));
    if (d[DSZ_OVERFLOW]) return lagpm_fail(ctx, LAGPM_E_STATE, "the last build overflowed its node arrays");
    const size_t nn = std::min<size_t>(d[DSZ_NODES], box->node_cap);
    *nnodes = nn;
    if (cap < nn) return lagpm_fail(ctx, LAGPM_E_INVAL, "the arrays hold fewer nodes than the tree has (see *nnodes)");
    // the records in the nodes' pre-order
    std::vector<uint32_t> rop(nn);
    RCHK(lagpm_d2h(ctx, rop.data(), box->nd_rop, nn * sizeof(uint32_t), box->st));
    if (info) {
        std::vector<int4> link(nn);
        std::vector<int> lev(nn);
        RCHK(lagpm_d2h(ctx, link.data(), box->nd_link, nn * sizeof(int4), box->st));
        RCHK(lagpm_d2h(ctx, lev.data(), box->nd_lev, nn * sizeof(int), box->st));
        for (size_t v = 0; v < nn; v++) {
            const int4 a = link[rop[v]];
            info[4 * v] = a.x; info[4 * v + 1] = a.y; info[4 * v + 2] = a.w; info[4 * v + 3] = lev[rop[v]] & 255;
        }
    }
    if (order) RCHK(lagpm_d2h(ctx, order, box->id, box->np * sizeof(uint32_t), box->st));
    if (!com && !quad) return LAGPM_OK;
    const double mass = box->p.mass;
    if (box->p.precision == LAGPM_PREC_FP64) {
        std::vector<double> t(12 * nn);
        RCHK(lagpm_d2h(ctx, t.data(), box->nd_d, t.size() * sizeof(double), box->st));
        for (size_t v = 0; v < nn; v++) {
            const double* a = &t[12 * (size_t)rop[v]];
            if (com) { com[4 * v] = a[0]; com[4 * v + 1] = a[1]; com[4 * v + 2] = a[2]; com[4 * v + 3] = a[3] * mass; }
            if (quad) {
                for (int k = 0; k < 7; k++) quad[8 * v + k] = a[4 + k] * mass;
                quad[8 * v + 7] = a[11];
            }
        }
        return LAGPM_OK;
    }
    std::vector<float4> c(nn), q0(nn), q1(nn);
    RCHK(lagpm_d2h(ctx, c.data(), box->nd_geo, nn * sizeof(float4), box->st));
    RCHK(lagpm_d2h(ctx, q0.data(), box->nd_q0, nn * sizeof(float4), box->st));
    RCHK(lagpm_d2h(ctx, q1.data(), box->nd_q1, nn * sizeof(float4), box->st));
    const double s = lagpm_tree_scale(box), s2 = s * s;
    for (size_t v = 0; v < nn; v++) {
        const size_t r = rop[v];
        if (com) {
            com[4 * v] = c[r].x / s; com[4 * v + 1] = c[r].y / s; com[4 * v + 2] = c[r].z / s;
            com[4 * v + 3] = q1[r].w * mass;
        }
        if (quad) {
            // (the record holds half the trace and the mass beside the quadrupole, rmax beside the centre)
            const double q[7] = {q0[r].x, q0[r].y, q0[r].z, q0[r].w, q1[r].x, q1[r].y, 2.0 * q1[r].z};
            for (int k = 0; k < 7; k++) quad[8 * v + k] = q[k] * mass / s2;
            quad[8 * v + 7] = c[r].w / s;
        }
    }
    return LAGPM_OK;
}
