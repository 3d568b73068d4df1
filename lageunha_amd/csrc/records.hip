// records.hip — GOTPM particle records on the device: decoding on upload (XofP/YofP/ZofP,
// eunha.h:1212, 1228-1232) and its inverse on download.
//
// A record is 32 bytes (dmparticletype under GOTPM + XYZDBL, eunha.h:389-399): u64 index|flag, f32
// displacement from the lattice site, f32 velocity. The host moves whole records and the device
// turns them into the box's FP64 arrays: one pass over HBM, where the same loop on one host thread
// (three fmod and three 64-bit divisions a record) took most of an upload.
#include "lagpm_internal.h"

namespace {

// one record as two 16-byte words
struct rec32 {
    ulonglong2 a;  // index|flag, (x, y)
    ulonglong2 b;  // (z, vx), (vy, vz)
};
static_assert(sizeof(rec32) == 32, "GOTPM particle is 32 bytes");

__device__ inline float lo_f(unsigned long long w) { return __uint_as_float((uint32_t)w); }
__device__ inline float hi_f(unsigned long long w) { return __uint_as_float((uint32_t)(w >> 32)); }

// lattice site of the low 56 bits of the index word: idx = i + n (j + n k)
__device__ inline void lattice_site(unsigned long long u4if, uint32_t n, double s[3]) {
    const unsigned long long idx = (u4if << 8) >> 8;  // PINDX, eunha.h:1212
    if (idx <= 0xffffffffull) {  // 32-bit divisions (64-bit ones are a software loop)
        const uint32_t q = (uint32_t)idx, r = q / n;
        s[0] = (double)(q - r * n);
        s[1] = (double)(r % n);
        s[2] = (double)(r / n);
    } else {
        const unsigned long long r = idx / n;
        s[0] = (double)(idx - r * n);
        s[1] = (double)(r % n);
        s[2] = (double)(r / n);
    }
}

// XofP = fmod(dx + i + nx, nx), then wrapped into [0, nx) as every upload is (a displacement below
// -nx leaves a negative remainder)
__device__ inline double decode_pos(float d, double site, double L) {
    double v = fmod((double)d + site + L, L);
    if (v < 0) v += L;
    if (v >= L) v = 0.0;
    return v;
}

// Bound by HBM: 32 bytes read and 52 written a record (the copy over PCIe takes longer). An upload of
// 2.1M records: 90 ms with the host loop and the copies of its 48 bytes a record, 1.7 ms with this.
__global__ void __launch_bounds__(256) decode_records_kernel(const rec32* __restrict__ rec, size_t first, size_t count, uint32_t n,
                                                             double* __restrict__ x, double* __restrict__ y, double* __restrict__ z,
                                                             double* __restrict__ vx, double* __restrict__ vy,
                                                             double* __restrict__ vz, uint32_t* __restrict__ id) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    const ulonglong2 a = rec[t].a, b = rec[t].b;
    double s[3];
    lattice_site(a.x, n, s);
    const double L = (double)n;
    const size_t i = first + t;
    x[i] = decode_pos(lo_f(a.y), s[0], L);
    y[i] = decode_pos(hi_f(a.y), s[1], L);
    z[i] = decode_pos(lo_f(b.x), s[2], L);
    vx[i] = (double)hi_f(b.x);
    vy[i] = (double)lo_f(b.y);
    vz[i] = (double)hi_f(b.y);
    id[i] = (uint32_t)i;
}

// the displacement from the record's own lattice site, taken as the periodic image nearest to it
// ([-n/2, n/2)), so XofP of the record gives the position back
__device__ inline uint32_t encode_pos(double pos, double site, double L) {
    const double h = 0.5 * L;
    double d = fmod(pos - site, L);
    if (d >= h) d -= L;
    if (d < -h) d += L;
    return __float_as_uint((float)d);
}

struct rec_quarters {
    uint32_t* p[4];  // records of 8 words, `q` of them in each
    uint32_t q;
};
// Particle i of the box's order is record id[i]: its index word is read there and the fields beside
// it are written (POS: displacement and velocity, otherwise the velocity alone). A record is half a
// 64-byte sector, so a particle touches one sector of the records however they are ordered.
template <bool POS>
__global__ void __launch_bounds__(256) encode_records_kernel(rec_quarters Q, size_t np, uint32_t n, const double* __restrict__ x,
                                                             const double* __restrict__ y, const double* __restrict__ z,
                                                             const double* __restrict__ vx, const double* __restrict__ vy,
                                                             const double* __restrict__ vz, const uint32_t* __restrict__ id) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const uint32_t r = id[i], k = r / Q.q;
    uint32_t* rec = Q.p[k] + 8 * (size_t)(r - k * Q.q);
    const uint32_t ux = __float_as_uint((float)vx[i]), uy = __float_as_uint((float)vy[i]), uz = __float_as_uint((float)vz[i]);
    if constexpr (POS) {
        const unsigned long long u4if = *reinterpret_cast<const unsigned long long*>(rec);
        double s[3];
        lattice_site(u4if, n, s);
        const double L = (double)n;
        rec[2] = encode_pos(x[i], s[0], L);
        rec[3] = encode_pos(y[i], s[1], L);
        rec[4] = encode_pos(z[i], s[2], L);
    }
    rec[5] = ux;
    rec[6] = uy;
    rec[7] = uz;
}

// the caller's records as copies to and from the scratch arrays
size_t quarters(lagpm_box* box, const void* dm_bp, lagpm_segment seg[4]) {
    static_assert(LAGPM_ARRAY_PAD * 8 >= 32, "a quarter rounded up fits its scratch array");
    const size_t np = box->np, q = (np + 3) / 4;
    size_t k = 0;
    for (size_t first = 0; first < np; k++, first += q)
        seg[k] = {box->alt[k], (char*)const_cast<void*>(dm_bp) + first * sizeof(rec32), std::min(q, np - first) * sizeof(rec32)};
    return k;
}

unsigned grid_of(size_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// The records pass through four of the box's scratch arrays (alt, free between sorts), a quarter of
// them each: their 8 bytes a particle hold the quarter's 32 bytes a record.
int lagpm_upload_records(lagpm_ctx* ctx, lagpm_box* box, const void* dm_bp) {
    const size_t q = (box->np + 3) / 4;
    lagpm_segment seg[4];
    const size_t nseg = quarters(box, dm_bp, seg);
    RCHK(lagpm_copy_segments(ctx, seg, nseg, false, box->st));
    for (size_t k = 0; k < nseg; k++) {
        const size_t cnt = seg[k].bytes / sizeof(rec32);
        hipLaunchKernelGGL(decode_records_kernel, dim3(grid_of(cnt)), dim3(256), 0, box->st, (const rec32*)box->alt[k], k * q, cnt,
                           (uint32_t)box->p.n, box->x, box->y, box->z, box->vx, box->vy, box->vz, box->id);
        HIPCHK(ctx, hipGetLastError());
    }
    return LAGPM_OK;
}

// The caller's records (their index words name the lattice sites) go to the device, get their fields
// there and come back whole: two copies at PCIe rate, where copying six FP64 arrays back and filling
// the records on one host thread took 39 ms for 2.1M records (this: 3.3 ms).
int lagpm_download_records(lagpm_ctx* ctx, lagpm_box* box, void* dm_bp, bool positions) {
    const size_t np = box->np, q = (np + 3) / 4;
    rec_quarters Q;
    Q.q = (uint32_t)q;
    for (int k = 0; k < 4; k++) Q.p[k] = reinterpret_cast<uint32_t*>(box->alt[k]);
    lagpm_segment seg[4];
    const size_t nseg = quarters(box, dm_bp, seg);
    RCHK(lagpm_copy_segments(ctx, seg, nseg, false, box->st));
    auto kern = positions ? encode_records_kernel<true> : encode_records_kernel<false>;
    hipLaunchKernelGGL(kern, dim3(grid_of(np)), dim3(256), 0, box->st, Q, np, (uint32_t)box->p.n, box->x, box->y, box->z, box->vx,
                       box->vy, box->vz, box->id);
    HIPCHK(ctx, hipGetLastError());
    return lagpm_copy_segments(ctx, seg, nseg, true, box->st);
}
