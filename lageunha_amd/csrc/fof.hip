// fof.hip — PreFoF halo-candidate flags on the device (Cosmos/PreFoF.c:207-386, OST/fof.c:190-293).
//
// The reference bins particles into cells of width 4 (Cosmos/BasicCell.h:1), grows friends-of-
// friends groups inside each cell alone with a per-cell tree (pnew_fof_link), and keeps every
// group that lies within the link of a cell face or has at least FOF_MINNUM members
// (CountHaloCandidates). The groups are the connected components of the link graph, so here:
//   1. each particle gets a key (cell, sub-cell) and the particles are radix-sorted by it (a cell's
//      particles, and each sub-cell's, are contiguous). A sub-cell's diagonal is shorter than the
//      link, so its particles are one set from the start;
//   2. one thread per particle searches the sub-cells within the link of it, in its own cell, for one
//      linked partner in each that is not in its set yet, and joins the two in a lock-free
//      union-find (roots are only ever hooked under smaller roots);
//   3. per group (at its root): member count, by atomics over its sub-cells, and whether a member
//      lies within the link of a cell face (the group's bounds are compared with the same limits);
//      then the flag rule.
// Pair distances and bounds are FP64 and use the reference's operations (relative coordinates
// X - 4*ix, sqrt(dx*dx + dy*dy + dz*dz) <= link, this file is built without FMA contraction), so
// the flags are the reference's bit for bit.
#include <vector>

#include "lagpm_internal.h"
#include "wave_ops.h"

namespace {

constexpr int FOF_SUB_MAX = 1024;  // sub-cells per cell edge at most (30 key bits)

__device__ inline uint32_t par_load(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void par_store(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Root of x with path halving. Every parent is smaller than its child (hooks put the larger root
// under the smaller one; halving stores an ancestor), so the walk strictly decreases and ends.
__device__ inline uint32_t uf_root(uint32_t* par, uint32_t x) {
    while (true) {
        const uint32_t p = par_load(par + x);
        if (p == x) return x;
        const uint32_t g = par_load(par + p);
        if (g == p) return p;
        par_store(par + x, g);
        x = g;
    }
}
// Joins the sets of a and b. A failed hook means another thread hooked that root first (a
// successful operation elsewhere), so the retries are bounded by the number of hooks.
__device__ inline void uf_unite(uint32_t* par, uint32_t a, uint32_t b) {
    a = uf_root(par, a);
    b = uf_root(par, b);
    while (a != b) {
        if (a < b) {
            const uint32_t t = a;
            a = b;
            b = t;
        }
        const uint32_t old = atomicCAS(par + a, a, b);
        if (old == a) return;
        a = uf_root(par, old);
        b = uf_root(par, b);
    }
}

struct fof_grid {
    uint32_t mx;  // cells per edge: ceil(n / 4)
    int k;        // sub-cells per cell edge
    int bits;     // key bits of a sub-cell number
    int reach;    // linked particles are at most this many sub-cells apart along an axis
    double kf;    // k / 4
    uint64_t ncell;
    double link;
    double wide;  // the link, and a margin far above the rounding of the sub-cell bounds
};

__device__ inline int sub_of(double r, const fof_grid& G) {
    return (int)fmin(fmax(r * G.kf, 0.0), (double)(G.k - 1));
}

struct fof_pos {  // relative positions in sorted order
    double *__restrict__ x, *__restrict__ y, *__restrict__ z;
};

__device__ inline uint32_t cell_of(double X, uint32_t mx) {
    const uint32_t c = (uint32_t)(X / 4.0);  // PreFoF.c:326-328 (X / 4 is exact)
    return c < mx ? c : mx - 1;
}

__global__ void fof_key_kernel(const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
                               size_t np, fof_grid G, uint64_t* __restrict__ key, uint32_t* __restrict__ val) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const double P[3] = {x[i], y[i], z[i]};
    uint32_t c[3], s[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        c[a] = cell_of(P[a], G.mx);
        s[a] = (uint32_t)sub_of(P[a] - 4.0 * (double)c[a], G);
    }
    uint64_t cell = (uint64_t)c[0] + (uint64_t)G.mx * ((uint64_t)c[1] + (uint64_t)G.mx * (uint64_t)c[2]);
    // a particle without a position is linked to none: such go into one more cell, after the others
    if (!(P[0] == P[0] && P[1] == P[1] && P[2] == P[2])) cell = G.ncell;
    const uint64_t sub = (uint64_t)s[0] + (uint64_t)G.k * ((uint64_t)s[1] + (uint64_t)G.k * (uint64_t)s[2]);
    key[i] = (cell << G.bits) | sub;
    val[i] = (uint32_t)i;
}

__device__ inline uint32_t lower_bound_key(const uint64_t* __restrict__ K, uint32_t lo, uint32_t hi, uint64_t v) {
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (K[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// first sorted position of every cell c in [0, ncell + 1] (start[ncell + 1] = np)
__global__ void fof_cellstart_kernel(const uint64_t* __restrict__ key, uint32_t np, uint64_t ncell, int bits,
                                     uint32_t* __restrict__ start) {
    const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c > ncell + 1) return;
    start[c] = lower_bound_key(key, 0, np, c << bits);
}

// Positions relative to the cell corner (Dump2FoFPtl, PreFoF.c:38-54) in sorted order, and the set-up
// of the union-find: the parent of a particle is the first one of its sub-cell (CLUMP), or itself.
// end[h] is the end of the sub-cell that begins at h, cnt[h] its members.
template <bool CLUMP>
__global__ void fof_gather_kernel(const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
                                  const uint64_t* __restrict__ key, const uint32_t* __restrict__ val, uint32_t np,
                                  fof_grid G, const uint32_t* __restrict__ start, fof_pos r, uint32_t* __restrict__ par,
                                  uint32_t* __restrict__ end, uint32_t* __restrict__ cnt, uint8_t* __restrict__ edge) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const uint32_t i = val[p];
    const double X = x[i], Y = y[i], Z = z[i];
    r.x[p] = X - 4.0 * (double)cell_of(X, G.mx);
    r.y[p] = Y - 4.0 * (double)cell_of(Y, G.mx);
    r.z[p] = Z - 4.0 * (double)cell_of(Z, G.mx);
    edge[p] = 0;
    const uint64_t kp = key[p];
    uint32_t head = p;
    const bool set = CLUMP && (kp >> G.bits) < G.ncell;
    if (set && p > 0 && key[p - 1] == kp) head = lower_bound_key(key, start[kp >> G.bits], p, kp);
    par[p] = head;
    if (!set || p + 1 == np || key[p + 1] != kp) {
        end[head] = p + 1;
        cnt[head] = p + 1 - head;
    }
}

__device__ inline bool linked(double px, double py, double pz, const fof_pos& r, uint32_t q, double link) {
    const double ex = fabs(px - r.x[q]), ey = fabs(py - r.y[q]), ez = fabs(pz - r.z[q]);
    return sqrt(ex * ex + ey * ey + ez * ez) <= link;  // OST/fof.c:272-276
}

// Distance from v to the sub-cells' slab t along one axis.
__device__ inline double slab_dist(double v, int t, const fof_grid& G) {
    return fmax(fmax((double)t / G.kf - v, v - (double)(t + 1) / G.kf), 0.0);
}

// Each unordered pair of sub-cells is searched from the lower one. The sub-cells of one row (fixed
// y and z) are consecutive in the sorted order, so a row costs one binary search, nearest rows
// first: by the time a halo's thread comes to the far ones their sub-cells are mostly in its set
// already, and are passed over whole.
// CLUMP: a sub-cell is one set, so one linked partner in it is enough. Testing every pair of
// sub-cells one link wide (in dense halos 10^4 tests a thread) took 5.9 ms for 2.1 million
// particles at a link of 0.2 with 30 % of them in halos; this takes 0.58 ms, of which the searches alone
// (no halos) are 0.12 and the rest is the unions' dependent loads.
template <bool CLUMP>
__global__ void fof_link_kernel(const uint64_t* __restrict__ key, fof_pos r,
                                const uint32_t* __restrict__ start, const uint32_t* __restrict__ end, uint32_t np, fof_grid G,
                                uint32_t* __restrict__ par) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const uint64_t kp = key[p];
    const uint64_t cell = kp >> G.bits, cellbits = cell << G.bits;
    if (cell == G.ncell) return;
    const uint32_t k = (uint32_t)G.k, sub = (uint32_t)(kp - cellbits);
    const int sy = (int)((sub / k) % k), sz = (int)(sub / (k * k));
    const uint32_t ce = start[cell + 1];
    const double px = r.x[p], py = r.y[p], pz = r.z[p];
    // an ancestor of p (ancestors stay ancestors): a partner whose parent is it is
    // already in p's set, which saves the two root searches of a union
    uint32_t rp = uf_root(par, p);
    auto join = [&](uint32_t q) {
        if (par_load(par + q) == rp) return;
        uf_unite(par, p, q);
        rp = uf_root(par, p);
    };
    // the sub-cells along x that p's link reaches
    const int x0 = sub_of(px - G.wide, G), x1 = sub_of(px + G.wide, G);
    for (int ring = 0; ring <= G.reach; ring++)
        for (int dz = 0; dz <= ring; dz++) {
            const int tz = sz + dz;
            if (tz >= G.k) break;
            for (int dy = dz ? -ring : ring; dy <= ring; dy++) {
                if (dz < ring && dy > -ring && dy < ring) dy = ring;
                const int ty = sy + dy;
                if (ty < 0 || ty >= G.k) continue;
                const uint32_t row = k * ((uint32_t)ty + k * (uint32_t)tz);
                uint32_t q;
                if (ring == 0) {
                    // p's own row: from the next particle on, or the next sub-cell where p's is one set
                    q = p + 1;
                    if (CLUMP && q < ce && key[q] == kp) q = end[lower_bound_key(key, start[cell], p, kp)];
                } else {
                    const double oy = slab_dist(py, ty, G), oz = slab_dist(pz, tz, G);
                    if (oy * oy + oz * oz > G.wide * G.wide) continue;
                    q = lower_bound_key(key, p + 1, ce, cellbits + row + (uint32_t)x0);
                }
                const uint64_t last = cellbits + row + (uint32_t)x1;
                while (q < ce && key[q] <= last) {
                    if constexpr (CLUMP) {
                        // q begins a sub-cell
                        const uint32_t e = end[q];
                        uint32_t j = q;
                        if (par_load(par + q) != rp)
                            for (; j < e; j++) {
                                // other threads may have joined the two meanwhile
                                if (((j - q) & 63u) == 0u && uf_root(par, q) == (rp = uf_root(par, rp))) break;
                                if (linked(px, py, pz, r, j, G.link)) {
                                    join(q);
                                    break;
                                }
                            }
                        q = e;
                    } else {
                        if (linked(px, py, pz, r, q, G.link)) join(q);
                        q++;
                    }
                }
            }
        }
}

// Only sub-cells that are not their group's root add to its count (a halo's 10^5 members are some 10^3 of
// them, one atomic a wave and group), and only members within the link of a cell face mark it. Bounds
// reduced at the roots by seven atomics a member took 0.46 ms (link 0.2, 2.1 million particles,
// 30 % in halos), an atomic for each sub-cell 0.18 (those of the largest halos wait for each other), this 0.036.
template <bool CLUMP>
__global__ void fof_stats_kernel(const uint64_t* __restrict__ key, fof_pos r, const uint32_t* __restrict__ end, uint32_t np,
                                 fof_grid G, uint32_t* __restrict__ par, uint32_t* __restrict__ cnt,
                                 uint8_t* __restrict__ edge) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = p < np;
    auto in = [&](double v) { return v > G.link && v < 4.0 - G.link; };  // CountHaloCandidates, PreFoF.c:238-251
    const bool inside = !valid || (in(r.x[p]) && in(r.y[p]) && in(r.z[p]));
    const bool head = valid && (!CLUMP || p == 0 || key[p - 1] != key[p]);
    uint32_t g = p;
    if (!inside || head) g = uf_root(par, p);
    if (!inside) edge[g] = 1;
    const int n = head && g != p ? (int)(end[p] - p) : 0;
    // one atomic for the wave's sub-cells of one group: the sorted order puts a halo's together
    unsigned long long left = __ballot(n > 0);
    while (left) {
        const int first = __ffsll(left) - 1;
        const uint32_t g0 = (uint32_t)__builtin_amdgcn_readlane((int)g, first);
        const bool same = n > 0 && g == g0;
        int sum;
        (void)lagpm_wave::wave_excl_scan(same ? n : 0, threadIdx.x & 63, sum);
        if ((int)(threadIdx.x & 63) == first) atomicAdd(cnt + g0, (uint32_t)sum);
        left &= ~__ballot(same);
    }
}

// a group inside [link, 4 - link) on every axis is kept only with minnum members or more; any other
// group is kept
__global__ void fof_flag_kernel(const uint32_t* __restrict__ val, const uint32_t* __restrict__ id, uint32_t np,
                                uint32_t* __restrict__ par, const uint32_t* __restrict__ cnt, const uint8_t* __restrict__ edge,
                                uint32_t minnum, uint8_t* __restrict__ flag) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const uint32_t g = uf_root(par, p);
    flag[id[val[p]]] = (uint8_t)(edge[g] || cnt[g] >= minnum);
}

unsigned grid_of(size_t n, int t) { return (unsigned)std::max<size_t>(1, (n + t - 1) / t); }

struct dev_buf {
    void* p = nullptr;
    ~dev_buf() {
        if (p) (void)hipFree(p);
    }
};

}  // namespace

extern "C" int lagpm_prefof(lagpm_ctx* ctx, lagpm_box* box, float fof_link, int minnum, uint8_t* flags,
                            size_t* nflagged) {
    if (!ctx || !box) return lagpm_fail(ctx, LAGPM_E_INVAL, "NULL argument");
    if (!box->uploaded) return lagpm_fail(ctx, LAGPM_E_STATE, "no particles uploaded");
    if (!(fof_link > 0.0f) || !(fof_link < 1e30f)) return lagpm_fail(ctx, LAGPM_E_INVAL, "fof_link must be positive and finite");
    if (minnum < 1) return lagpm_fail(ctx, LAGPM_E_INVAL, "minnum must be at least 1");
    const size_t np = box->np;
    if (nflagged) *nflagged = 0;
    if (np == 0) return LAGPM_OK;
    HIPCHK(ctx, hipSetDevice(ctx->device));
    const double link = (double)fof_link;
    fof_grid G;
    G.mx = (uint32_t)((box->p.n + 3) / 4);
    G.link = link;
    G.wide = link + 1e-9 * (4.0 + link);
    // The fewest sub-cells whose diagonal is below the link by a margin far above rounding (1e-15 of
    // 4). Where that takes more than the key holds (links below 0.0068) the sub-cells stay the
    // particles' own sets, strictly wider than the link.
    const double need = std::ceil(4.0 * std::sqrt(3.0) / link * (1.0 + 1e-9));
    const bool clump = need <= FOF_SUB_MAX;
    G.k = clump ? std::max(1, (int)need) : FOF_SUB_MAX / 2;
    G.kf = (double)G.k / 4.0;
    G.reach = (int)std::min((double)G.k, std::floor(G.wide * G.kf) + 1.0);
    const uint64_t ncell = G.ncell = (uint64_t)G.mx * G.mx * G.mx;
    int cbits = 1;
    while ((1ull << cbits) < ncell + 1) cbits++;
    G.bits = 1;
    while ((1ull << G.bits) < (uint64_t)G.k * G.k * G.k) G.bits++;
    const int bits = cbits + G.bits;
    hipStream_t st = box->st;
    // The scratch is the box's other particle set (52 bytes a particle, which the next sort writes
    // anew) and its sort scratch: allocating and freeing 93 bytes a particle took 0.4 ms of a
    // call with 2.1 million particles.
    fof_pos r{box->alt[0], box->alt[1], box->alt[2]};
    uint64_t* key = (uint64_t*)box->alt[3];
    uint64_t* key2 = (uint64_t*)box->alt[4];
    uint32_t* par = (uint32_t*)box->alt[5];
    uint32_t* val = par + np;
    uint32_t* val2 = box->id_alt;
    hipLaunchKernelGGL(fof_key_kernel, dim3(grid_of(np, 256)), dim3(256), 0, st, box->x, box->y, box->z, np, G, key, val);
    HIPCHK(ctx, hipGetLastError());
    bool in_alt = false;
    RCHK(lagpm_radix_sort_pairs(ctx, st, box->scan_tmp, key, key2, val, val2, np, bits, &in_alt));
    if (in_alt) {
        std::swap(key, key2);
        std::swap(val, val2);
    }
    // what the sort leaves free: a key buffer (8 bytes a particle), a value buffer (4), its tables
    uint32_t* end = (uint32_t*)key2;
    uint32_t* cnt = end + np;
    uint8_t* edge = (uint8_t*)val2;
    uint8_t* dflag = edge + np;
    dev_buf mem;
    uint32_t* start = box->scan_tmp;
    if (4 * (ncell + 2) > box->scan_tmp_bytes) {  // few particles in a large box
        if (hipMalloc(&mem.p, 4 * (ncell + 2)) != hipSuccess) {
            (void)hipGetLastError();
            return lagpm_fail(ctx, LAGPM_E_NOMEM, "PreFoF scratch (" + std::to_string(4 * (ncell + 2)) + " bytes) does not fit");
        }
        start = (uint32_t*)mem.p;
    }
    hipLaunchKernelGGL(fof_cellstart_kernel, dim3(grid_of(ncell + 2, 256)), dim3(256), 0, st, key, (uint32_t)np, ncell,
                       G.bits, start);
    HIPCHK(ctx, hipGetLastError());
    const dim3 grid(grid_of(np, 256)), blk(256);
    const uint32_t m = (uint32_t)np;
    hipLaunchKernelGGL(clump ? fof_gather_kernel<true> : fof_gather_kernel<false>, grid, blk, 0, st, box->x, box->y, box->z, key,
                       val, m, G, start, r, par, end, cnt, edge);
    HIPCHK(ctx, hipGetLastError());
    hipLaunchKernelGGL(clump ? fof_link_kernel<true> : fof_link_kernel<false>, grid, blk, 0, st, key, r, start, end, m, G, par);
    HIPCHK(ctx, hipGetLastError());
    hipLaunchKernelGGL(clump ? fof_stats_kernel<true> : fof_stats_kernel<false>, grid, blk, 0, st, key, r, end, m, G, par, cnt,
                       edge);
    HIPCHK(ctx, hipGetLastError());
    hipLaunchKernelGGL(fof_flag_kernel, grid, blk, 0, st, val, box->id, m, par, cnt, edge, (uint32_t)minnum, dflag);
    HIPCHK(ctx, hipGetLastError());
    std::vector<uint8_t> h(flags ? 0 : np);
    if (!flags) flags = h.data();
    RCHK(lagpm_d2h(ctx, flags, dflag, np, st));
    size_t c = 0;
    for (size_t i = 0; i < np; i++) c += flags[i];
    if (nflagged) *nflagged = c;
    return LAGPM_OK;
}
