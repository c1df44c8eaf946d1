// Pixel values of a galaxy catalogue: weighted galaxy counts per cell and
// y = B^T x with x_a = (N_a - Nbar_a)/sqrt(Nbar_a) -- the dot stage
// (src/dot.cpp:105-157).
//
// Counting.  The reference adds each galaxy's weight into counts[a] in
// catalogue order (src/dot.cpp:124-128), so the per-cell sums are left folds
// whose rounding depends on that order.  Here every galaxy gets its bin key
// (cell number, or Ncells for "outside every cell"), a stable radix sort
// groups the keys while keeping catalogue order inside each group, and one
// thread per bin folds its group in that order: the counts are bit-identical
// to the sequential loop.  Catalogues are taken in chunks of CHUNK galaxies;
// a chunk's fold starts from the previous chunk's count, so chunking does not
// change a bit either.
//
// Two defects of the reference loop are not reproduced: a galaxy in grid cell
// e = 0 is counted as outside (`e > 0`, src/dot.cpp:127), and a galaxy in a
// grid position with no cell indexes counts[-1].  Here e >= 0 is inside, and
// grid positions without a cell count as outside.
#include <rocprim/device/device_radix_sort.hpp>

#include "common.h"

namespace opsec {

struct DotState {
    int* d_map = nullptr;          // grid index -> cell number, -1 for none
    size_t cap_map = 0;
    float4* d_gal = nullptr;       // one chunk of galaxies
    size_t cap_gal = 0;
    uint32_t* d_key[2] = {nullptr, nullptr};
    size_t cap_key[2] = {0, 0};
    float* d_w[2] = {nullptr, nullptr};
    size_t cap_w[2] = {0, 0};
    void* d_tmp = nullptr;         // radix-sort temporary storage
    size_t cap_tmp = 0;
    double* d_counts = nullptr;    // Ncells + 1
    size_t cap_counts = 0;
    double* d_x = nullptr;         // Ncells
    size_t cap_x = 0;
    double* d_y = nullptr;         // Nmodes
    size_t cap_y = 0;
};

namespace {

constexpr int64_t CHUNK = int64_t(1) << 26;

struct GridGeom {
    double lo1, hi1, lo2, hi2, lo3, hi3;
    int n1, n2, n3;
};

// floor(n (x - lo)/(hi - lo)) in the operation order of Survey::GetGridIndex
// (src/Survey.cpp:93-101); -1 outside [0, n).  The comparison is made on the
// floored double, which also sends NaN and out-of-int-range values outside.
__device__ __forceinline__ int grid_coord(float x, double lo, double hi, int n) {
    double t = floor((double)n * ((double)x - lo) / (hi - lo));
    return (t >= 0.0 && t < (double)n) ? (int)t : -1;
}

__global__ void fill_int_kernel(int* p, int64_t n, int v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// cellmap[e] = a for every cell; when two cells share a grid position the
// larger cell number wins, as the reference's in-order loop leaves it
// (src/dot.cpp:106-115).
__global__ void cellmap_kernel(const int* __restrict__ cellidx, int ncells, int n2, int n3, int* map) {
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= ncells) return;
    int64_t e = ((int64_t)cellidx[3 * a] * n2 + cellidx[3 * a + 1]) * n3 + cellidx[3 * a + 2];
    atomicMax(map + e, a);
}

__global__ void galaxy_keys_kernel(const float4* __restrict__ gal, int64_t n, GridGeom g,
                                   const int* __restrict__ map, uint32_t nbins_out,
                                   uint32_t* __restrict__ key, float* __restrict__ w) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 p = gal[i];
    int d1 = grid_coord(p.x, g.lo1, g.hi1, g.n1);
    int d2 = grid_coord(p.y, g.lo2, g.hi2, g.n2);
    int d3 = grid_coord(p.z, g.lo3, g.hi3, g.n3);
    uint32_t k = nbins_out;
    if (d1 >= 0 && d2 >= 0 && d3 >= 0) {
        int a = map[((int64_t)d1 * g.n2 + d2) * g.n3 + d3];
        if (a >= 0) k = (uint32_t)a;
    }
    key[i] = k;
    w[i] = p.w;
}

__device__ __forceinline__ int64_t lower_bound_u32(const uint32_t* __restrict__ k, int64_t n, uint32_t v) {
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        int64_t mid = (lo + hi) >> 1;
        if (k[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// counts[b] += w over bin b's galaxies, one by one in catalogue order.  Bins of
// more than LONG_BIN galaxies are listed for fold_long_kernel instead.
constexpr int LONG_BIN = 1024;
__global__ void fold_bins_kernel(const uint32_t* __restrict__ key, const float* __restrict__ w, int64_t n,
                                 int nbins, double* __restrict__ counts, int* __restrict__ longs) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbins) return;
    int64_t lo = lower_bound_u32(key, n, (uint32_t)b);
    int64_t hi = lower_bound_u32(key, n, (uint32_t)b + 1);
    if (lo == hi) return;
    if (hi - lo > LONG_BIN) {
        longs[1 + atomicAdd(longs, 1)] = b;
        return;
    }
    double s = counts[b];
    int64_t i = lo;
    for (; i + 8 <= hi; i += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = w[i + j];
#pragma unroll
        for (int j = 0; j < 8; j++) s += (double)v[j];
    }
    for (; i < hi; i++) s += (double)w[i];
    counts[b] = s;
}

// The same fold of a long bin (the galaxies outside the survey above all), one
// workgroup per bin, with the bits of the serial loop.  While the sum stays
// within one binade, s = k u with u = ulp(s) and k an integer in [2^52, 2^53),
// adding w >= 0 rounds k + w/u to the nearest integer, ties to even: k grows by
// an integer that depends on k only where w/u is a half-integer, and then only
// on its parity.  So an addition is a map (parity -> increment), such maps
// compose associatively, and a block of FOLD_BLOCK weights is composed by all
// threads at once; the sums within it only grow, so if the last is below 2^53
// all were.  Weights of 2^51 u and more are not composed: without them a block's
// increments stay below 2048 x 2^51 = 2^62 and no sum of them wraps.  Where a
// block fails (the sum leaves the binade, a weight is that large, negative or not
// finite, the sum is not positive and normal), the waves before the failing
// one are kept, that wave's weights are added one by one from LDS, and the next
// block starts behind them.
// Bound by the composition's latency per block: 542 000 galaxies of one bin (two
// million, a quarter of them outside the survey) take 424 us, 9.85 ms by one thread (a
// dependent FP64 addition and its load each).
constexpr int FOLD_THREADS = 512, FOLD_PER = 4, FOLD_BLOCK = FOLD_THREADS * FOLD_PER;
constexpr int FOLD_WAVES = FOLD_THREADS / 64, FOLD_WAVE = 64 * FOLD_PER;
constexpr double FOLD_STEP = 2251799813685248.0;   // 2^51
static_assert(FOLD_BLOCK <= 2048, "a block's increments, at most 2^51 each, and k < 2^53 stay below 2^63");
struct FoldMap {
    long long c0, c1;   // increment of an even, of an odd k
    // this addition (or block) first, then b
    __device__ __forceinline__ void then(const FoldMap& b) {
        c0 += (c0 & 1) ? b.c1 : b.c0;
        c1 += (c1 & 1) ? b.c0 : b.c1;   // an odd k moved by an odd step is even
    }
};
// The map of the lane O further on in its row of 16 (zero past the row's end).
template <int O>
__device__ __forceinline__ FoldMap row_next(const FoldMap& f) {
    auto mv = [](long long x) {
        const unsigned lo = __builtin_amdgcn_mov_dpp((unsigned)x, 0x100 | O, 0xF, 0xF, true);
        const unsigned hi = __builtin_amdgcn_mov_dpp((unsigned)((unsigned long long)x >> 32), 0x100 | O, 0xF, 0xF, true);
        return (long long)((unsigned long long)hi << 32 | lo);
    };
    return FoldMap{mv(f.c0), mv(f.c1)};
}
__global__ __launch_bounds__(FOLD_THREADS) void fold_long_kernel(const uint32_t* __restrict__ key,
                                                                 const float* __restrict__ w, int64_t n,
                                                                 double* __restrict__ counts,
                                                                 const int* __restrict__ longs) {
    __shared__ FoldMap part[2][FOLD_WAVES * 4];   // one per row of 16 lanes
    __shared__ int bad[2][FOLD_WAVES];
    __shared__ float buf[FOLD_WAVE];
    __shared__ double sh_s;
    if ((int)blockIdx.x >= longs[0]) return;
    const int b = longs[1 + blockIdx.x], t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t lo = lower_bound_u32(key, n, (uint32_t)b), hi = lower_bound_u32(key, n, (uint32_t)b + 1);
    double s = counts[b];
    float nx[FOLD_PER];
    auto load = [&](int64_t at) {
#pragma unroll
        for (int j = 0; j < FOLD_PER; j++) {
            const int64_t i = at + FOLD_PER * t + j;
            nx[j] = i < hi ? w[i] : 0.0f;   // adding 0 to a positive sum changes nothing
        }
    };
    load(lo);
    int ph = 0;
    for (int64_t at = lo; at < hi; ph ^= 1) {
        float v[FOLD_PER];
#pragma unroll
        for (int j = 0; j < FOLD_PER; j++) v[j] = nx[j];
        if (at + FOLD_BLOCK < hi) load(at + FOLD_BLOCK);
        const unsigned long long bits = __double_as_longlong(s);
        const int e = (int)(bits >> 52) - 1023;          // s in [2^e, 2^(e+1)) when it is positive and normal
        const bool normal = e > -800 && e < 800;         // (a negative sum has the sign in e: above 800)
        const long long k = (long long)((bits & 0xfffffffffffffull) | 0x10000000000000ull);
        FoldMap f{0, 0};
        bool ok = normal;
#pragma unroll
        for (int j = 0; j < FOLD_PER; j++) {
            const double q = ldexp((double)v[j], 52 - e);   // w / u, exact
            ok = ok && q >= 0.0 && q < FOLD_STEP;
            const double r = rint(q), d = q - r;
            FoldMap g;
            g.c0 = g.c1 = (long long)(ok ? r : 0.0);
            if (fabs(d) == 0.5) {   // tie: to the even neighbour of k + w/u
                const long long l = (long long)(ok ? q - 0.5 : 0.0);
                g.c0 = l + (l & 1);
                g.c1 = l + (~l & 1);
            }
            f.then(g);
        }
        f.then(row_next<1>(f));
        f.then(row_next<2>(f));
        f.then(row_next<4>(f));
        f.then(row_next<8>(f));
        const bool wave_bad = __ballot(!ok) != 0;
        if ((lane & 15) == 0) part[ph][wave * 4 + (lane >> 4)] = f;
        if (lane == 0) bad[ph][wave] = wave_bad;
        __syncthreads();
        // the whole block: its 32 rows, one per lane, composed like the lanes were
        {
            FoldMap F = lane < 4 * FOLD_WAVES ? part[ph][lane] : FoldMap{0, 0};
            const bool any = __ballot(lane < FOLD_WAVES && bad[ph][lane & (FOLD_WAVES - 1)]) != 0;
            F.then(row_next<1>(F));
            F.then(row_next<2>(F));
            F.then(row_next<4>(F));
            F.then(row_next<8>(F));
            long long kw = k;
#pragma unroll
            for (int i = 0; i < 4 * FOLD_WAVES; i += 16) {
                const long long c0 = __shfl(F.c0, i), c1 = __shfl(F.c1, i);
                kw += (kw & 1) ? c1 : c0;
            }
            if (!any && kw < 9007199254740992ll) {
                s = ldexp((double)kw, e - 52);
                at += FOLD_BLOCK;
                continue;
            }
        }
        // the sum after each wave's weights, up to the first wave that fails
        long long k1 = k;
        int good = 0;
        for (; good < FOLD_WAVES - 1; good++) {   // the last one if no earlier
            long long kw = k1;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const FoldMap& F = part[ph][good * 4 + i];
                kw += (kw & 1) ? F.c1 : F.c0;
            }
            if (bad[ph][good] || kw >= 9007199254740992ll) break;
            k1 = kw;
        }
        if (good > 0) s = ldexp((double)k1, e - 52);
        if (wave == good)
#pragma unroll
            for (int j = 0; j < FOLD_PER; j++) buf[FOLD_PER * lane + j] = v[j];
        __syncthreads();
        at += good * FOLD_WAVE;
        if (t == 0 && at < hi) {
            const int m = (int)(hi - at < FOLD_WAVE ? hi - at : FOLD_WAVE);
            int i = 0;
            for (; i + 16 <= m; i += 16) {
                float x[16];
#pragma unroll
                for (int j = 0; j < 16; j++) x[j] = buf[i + j];
#pragma unroll
                for (int j = 0; j < 16; j++) s += (double)x[j];
            }
            for (; i < m; i++) s += (double)buf[i];
        }
        at += FOLD_WAVE;
        load(at);
        if (t == 0) sh_s = s;
        __syncthreads();
        s = sh_s;
    }
    if (t == 0) counts[b] = s;
}

// x_a = (N_a - Nbar_a)/sqrt(Nbar_a)  (src/dot.cpp:130-134)
__global__ void density_kernel(const double* __restrict__ counts, const double* __restrict__ nbar, int n,
                               double* __restrict__ x) {
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a < n) x[a] = (counts[a] - nbar[a]) / sqrt(nbar[a]);
}

// y_i = sum_a B_ia x_a: one 256-thread workgroup per mode.  Each thread folds
// a stride-256 subsequence, then a fixed LDS tree combines the 256 partials,
// so y does not depend on timing.
constexpr int GEMV_THREADS = 256;
__global__ __launch_bounds__(GEMV_THREADS) void modes_gemv_kernel(const double* __restrict__ B, int64_t ncells,
                                                                  const double* __restrict__ x,
                                                                  double* __restrict__ y) {
    __shared__ double part[GEMV_THREADS];
    const double* b = B + (int64_t)blockIdx.x * ncells;
    int t = threadIdx.x;
    double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    int64_t a = t;
    for (; a + 3 * GEMV_THREADS < ncells; a += 4 * GEMV_THREADS) {
        s0 += b[a] * x[a];
        s1 += b[a + GEMV_THREADS] * x[a + GEMV_THREADS];
        s2 += b[a + 2 * GEMV_THREADS] * x[a + 2 * GEMV_THREADS];
        s3 += b[a + 3 * GEMV_THREADS] * x[a + 3 * GEMV_THREADS];
    }
    for (; a < ncells; a += GEMV_THREADS) s0 += b[a] * x[a];
    part[t] = (s0 + s1) + (s2 + s3);
    __syncthreads();
    for (int h = GEMV_THREADS / 2; h > 0; h >>= 1) {
        if (t < h) part[t] += part[t + h];
        __syncthreads();
    }
    if (t == 0) y[blockIdx.x] = part[0];
}

unsigned blocks_for(int64_t n, int threads) { return (unsigned)((n + threads - 1) / threads); }

int ensure_dot(opsec_ctx* ctx) {
    if (!ctx->dot) ctx->dot = new DotState;
    return OPSEC_OK;
}

}  // namespace

void free_dot(opsec_ctx* ctx) {
    DotState* d = ctx->dot;
    if (!d) return;
    dev_free((void**)&d->d_map);
    dev_free((void**)&d->d_gal);
    for (int i = 0; i < 2; i++) {
        dev_free((void**)&d->d_key[i]);
        dev_free((void**)&d->d_w[i]);
    }
    dev_free(&d->d_tmp);
    dev_free((void**)&d->d_counts);
    dev_free((void**)&d->d_x);
    dev_free((void**)&d->d_y);
    delete d;
    ctx->dot = nullptr;
}

}  // namespace opsec

using namespace opsec;

extern "C" {


int opsec_count_galaxies(opsec_ctx* ctx, const opsec_galaxy* gals, int64_t ngals, int accumulate, double* counts) {
    if (!ctx) return OPSEC_EINVAL;
    if (ctx->ncells == 0) return set_error(ctx, OPSEC_ESTATE, "no survey uploaded");
    OPSEC_CHECK_ARG(ctx, counts, "no counts buffer");
    OPSEC_CHECK_ARG(ctx, ngals >= 0 && (gals || ngals == 0), "bad galaxy array");
    static_assert(sizeof(opsec_galaxy) == sizeof(float4), "galaxy record is four floats");
    OPSEC_HIP_TRY(ctx, hipSetDevice(ctx->device));
    int rc = ensure_dot(ctx);
    if (rc) return rc;
    DotState* d = ctx->dot;
    const SurveyDev& sv = ctx->sv;
    const int ncells = ctx->ncells, nbins = ncells + 1;
    const int64_t ngrid = (int64_t)sv.n1 * sv.n2 * sv.n3;

    if ((rc = dev_realloc(ctx, (void**)&d->d_map, &d->cap_map, (size_t)ngrid * 4))) return rc;
    if ((rc = dev_realloc(ctx, (void**)&d->d_counts, &d->cap_counts, (size_t)nbins * 8))) return rc;
    hipLaunchKernelGGL(fill_int_kernel, dim3(blocks_for(ngrid, 256)), dim3(256), 0, ctx->stream, d->d_map, ngrid, -1);
    hipLaunchKernelGGL(cellmap_kernel, dim3(blocks_for(ncells, 256)), dim3(256), 0, ctx->stream, ctx->d_cellidx,
                       ncells, sv.n2, sv.n3, d->d_map);
    OPSEC_HIP_TRY(ctx, hipGetLastError());
    if (accumulate)
        OPSEC_HIP_TRY(ctx, hipMemcpyAsync(d->d_counts, counts, (size_t)nbins * 8, hipMemcpyHostToDevice, ctx->stream));
    else
        OPSEC_HIP_TRY(ctx, hipMemsetAsync(d->d_counts, 0, (size_t)nbins * 8, ctx->stream));

    GridGeom g{sv.min1, sv.max1, sv.min2, sv.max2, sv.min3, sv.max3, sv.n1, sv.n2, sv.n3};
    unsigned end_bit = 1;
    while (end_bit < 32 && ((uint64_t)1 << end_bit) <= (uint64_t)ncells) end_bit++;

    const int64_t chunk_max = ngals < CHUNK ? ngals : CHUNK;
    if (chunk_max > 0) {
        if ((rc = dev_realloc(ctx, (void**)&d->d_gal, &d->cap_gal, (size_t)chunk_max * 16))) return rc;
        for (int i = 0; i < 2; i++) {
            if ((rc = dev_realloc(ctx, (void**)&d->d_key[i], &d->cap_key[i], (size_t)chunk_max * 4))) return rc;
            if ((rc = dev_realloc(ctx, (void**)&d->d_w[i], &d->cap_w[i], (size_t)chunk_max * 4))) return rc;
        }
        size_t tmp = 0;
        OPSEC_HIP_TRY(ctx, rocprim::radix_sort_pairs(nullptr, tmp, d->d_key[0], d->d_key[1], d->d_w[0], d->d_w[1],
                                                     (size_t)chunk_max, 0u, end_bit, ctx->stream));
        if ((rc = dev_realloc(ctx, &d->d_tmp, &d->cap_tmp, tmp))) return rc;
    }
    for (int64_t off = 0; off < ngals; off += CHUNK) {
        const int64_t n = (ngals - off) < CHUNK ? (ngals - off) : CHUNK;
        OPSEC_HIP_TRY(ctx, stream_copy(ctx, d->d_gal, gals + off, (size_t)n * 16, hipMemcpyHostToDevice));
        hipLaunchKernelGGL(galaxy_keys_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, d->d_gal, n, g,
                           d->d_map, (uint32_t)ncells, d->d_key[0], d->d_w[0]);
        OPSEC_HIP_TRY(ctx, hipGetLastError());
        size_t tmp = d->cap_tmp;
        OPSEC_HIP_TRY(ctx, rocprim::radix_sort_pairs(d->d_tmp, tmp, d->d_key[0], d->d_key[1], d->d_w[0], d->d_w[1],
                                                     (size_t)n, 0u, end_bit, ctx->stream));
        // at most n / LONG_BIN bins are long: their number, then their list, in the sort's
        // first key buffer (free again)
        int* longs = (int*)d->d_key[0];
        const int nlong = (int)std::min<int64_t>(nbins, n / (LONG_BIN + 1));
        hipLaunchKernelGGL(fill_int_kernel, dim3(1), dim3(64), 0, ctx->stream, longs, 1, 0);
        hipLaunchKernelGGL(fold_bins_kernel, dim3(blocks_for(nbins, 256)), dim3(256), 0, ctx->stream, d->d_key[1],
                           d->d_w[1], n, nbins, d->d_counts, longs);
        if (nlong > 0)
            hipLaunchKernelGGL(fold_long_kernel, dim3(nlong), dim3(FOLD_THREADS), 0, ctx->stream, d->d_key[1], d->d_w[1],
                               n, d->d_counts, longs);
        OPSEC_HIP_TRY(ctx, hipGetLastError());
    }
    OPSEC_HIP_TRY(ctx, hipMemcpyAsync(counts, d->d_counts, (size_t)nbins * 8, hipMemcpyDeviceToHost, ctx->stream));
    OPSEC_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return OPSEC_OK;
}

int opsec_pixel_values(opsec_ctx* ctx, const double* counts, double* x, double* y) {
    if (!ctx) return OPSEC_EINVAL;
    if (ctx->ncells == 0) return set_error(ctx, OPSEC_ESTATE, "no survey uploaded");
    if (ctx->nmodes == 0 || !ctx->d_B) return set_error(ctx, OPSEC_ESTATE, "no modes uploaded");
    OPSEC_CHECK_ARG(ctx, counts && y, "null counts or pixel buffer");
    OPSEC_HIP_TRY(ctx, hipSetDevice(ctx->device));
    int rc = ensure_dot(ctx);
    if (rc) return rc;
    DotState* d = ctx->dot;
    const int N = ctx->ncells, M = ctx->nmodes;
    if ((rc = dev_realloc(ctx, (void**)&d->d_counts, &d->cap_counts, (size_t)(N + 1) * 8))) return rc;
    if ((rc = dev_realloc(ctx, (void**)&d->d_x, &d->cap_x, (size_t)N * 8))) return rc;
    if ((rc = dev_realloc(ctx, (void**)&d->d_y, &d->cap_y, (size_t)M * 8))) return rc;
    OPSEC_HIP_TRY(ctx, hipMemcpyAsync(d->d_counts, counts, (size_t)N * 8, hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(density_kernel, dim3(blocks_for(N, 256)), dim3(256), 0, ctx->stream, d->d_counts, ctx->d_nbar,
                       N, d->d_x);
    hipLaunchKernelGGL(modes_gemv_kernel, dim3(M), dim3(GEMV_THREADS), 0, ctx->stream, ctx->d_B, (int64_t)N, d->d_x,
                       d->d_y);
    OPSEC_HIP_TRY(ctx, hipGetLastError());
    if (x) OPSEC_HIP_TRY(ctx, hipMemcpyAsync(x, d->d_x, (size_t)N * 8, hipMemcpyDeviceToHost, ctx->stream));
    OPSEC_HIP_TRY(ctx, hipMemcpyAsync(y, d->d_y, (size_t)M * 8, hipMemcpyDeviceToHost, ctx->stream));
    OPSEC_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return OPSEC_OK;
}

}  // extern "C"
