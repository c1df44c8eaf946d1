// FP64 / FP32 MFMA GEMM on k-contiguous operands: C[m][n] = sum_k A[m][k] B[n][k].
//
// Both operands are rows of T with 16-byte aligned pitches, and K is a whole
// number of 128-byte steps (nt_kpad); the columns between the real extent and
// the padded one are zero in both operands, so that an infinity or NaN in a row
// reaches only what its own products reach.  Rows
// beyond an operand's extent are clamped to its last row and their products
// dropped in the epilogue, so any M and N are taken.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "gemm.h"

namespace opsec {

constexpr int NT_BM = 128, NT_BN = 128;           // workgroup tile
constexpr int NT_STAGE = (NT_BM + NT_BN) * 128;   // bytes of one LDS stage: 128 rows x 128 bytes per operand
constexpr size_t NT_LDS = 2 * NT_STAGE;

// k values per step (128 bytes) and the padded extent / pitch of an operand row.
template <typename T>
constexpr int nt_bk() {
    return 128 / (int)sizeof(T);
}
template <typename T>
inline size_t nt_kpad(size_t k) {
    return (k + nt_bk<T>() - 1) / nt_bk<T>() * nt_bk<T>();
}
// 128 bytes more than the padded extent: a power-of-two pitch would put every
// row of a tile on the same L2 sets and HBM channels.
template <typename T>
inline size_t nt_pitch(size_t k) {
    return nt_kpad<T>(k) + nt_bk<T>();
}

// Position in an operand row of its k-th value, and k of a position, in the serial order
// of an FP32 product.  Lane group g of an MFMA takes the chunk 4 h + g of a step, so
// element e of it is MFMA e's: with k = 16 h + 4 e + g there, every MFMA adds four
// consecutive k, and a product is the chain of fused multiply-adds over k, the bits
// of any kernel that sums so.  Both operands of a product use the order or neither does.
__host__ __device__ __forceinline__ int nt_serial(int k) { return (k & ~15) | (k & 3) << 2 | (k >> 2 & 3); }

template <typename T>
struct NtMma;
template <>
struct NtMma<double> {
    typedef d4_t acc_t;
    typedef double vec_t __attribute__((ext_vector_type(2)));   // 16 bytes of consecutive k
    __device__ __forceinline__ static acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};
template <>
struct NtMma<float> {
    typedef f4_t acc_t;
    typedef f4_t vec_t;
    __device__ __forceinline__ static acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};

// Batches: z = band * nbat + b.  A is at b * a_bs + band * a_qs, B at
// band * b_qs + ((b + 1) >> 1) * b_bs: the transformed blocks of the Toeplitz
// projection (real and imaginary part of one frequency) share the B operand of
// their frequency.
template <typename T>
struct NtArgs {
    const T* A;
    size_t lda, a_bs, a_qs;
    int M;
    const T* B;
    size_t ldb, b_bs, b_qs;
    int N;
    int ksteps;            // K / nt_bk
    int nbat, nz;          // batches per band, nbat * bands
    bool serial = false;   // K in one piece: the operands are in the serial order
    // set by launch_nt_gemm
    int item0 = 0;         // first work item of the launch (item = z * tiles + tile)
    int nsplit = 1;        // split-K launch: its items, each in gridDim.x / nsplit parts
    T* ws = nullptr;       // split-K launch: the parts' accumulators
};

// Epilogues: base(band, b), then put(base, m, n, M, value), or put_in where inside(m0, n0, M)
// says that the whole tile is there (with put's tests and their loads for every element a
// tile of 209 k-steps took 1.8 % longer).
template <typename T, bool SERIAL>
struct NtRows {              // C[m * ld + n], n < nc, then zeros up to nw; SERIAL: in that order
    T* p;
    size_t ld, b_stride, q_stride;
    int nc, nw;
    __device__ __forceinline__ T* base(int q, int b) const { return p + q * q_stride + b * b_stride; }
    __device__ __forceinline__ bool inside(int m0, int n0, int M) const { return m0 + NT_BM <= M && n0 + NT_BN <= nc; }
    __device__ __forceinline__ void put_in(T* o, int m, int n, T v) const {
        o[(size_t)m * ld + (SERIAL ? nt_serial(n) : n)] = v;
    }
    __device__ __forceinline__ void put(T* o, int m, int n, int M, T v) const {
        if (m < M && n < nw) o[(size_t)m * ld + (SERIAL ? nt_serial(n) : n)] = n < nc ? v : (T)0;
    }
    static constexpr bool lower = false;
};
struct NtPacked {            // P[m (m + 1) / 2 + n] for n <= m: column m of a packed upper triangle
    double* p;
    size_t q_stride;
    __device__ __forceinline__ double* base(int q, int) const { return p + q * q_stride; }
    __device__ __forceinline__ bool inside(int m0, int n0, int M) const { return m0 + NT_BM <= M && n0 + NT_BN <= m0 + 1; }
    __device__ __forceinline__ void put_in(double* o, int m, int n, double v) const {
        o[(size_t)m * (m + 1) / 2 + n] = v;
    }
    __device__ __forceinline__ void put(double* o, int m, int n, int M, double v) const {
        if (m < M && n <= m) o[(size_t)m * (m + 1) / 2 + n] = v;
    }
    static constexpr bool lower = true;
};

// Tiles in groups of eight tile rows, column by column within a group, so that
// the 64 tiles resident on one XCD are about 8 x 8 and share their operands'
// rows in its L2.  lower: only the tiles of the lower triangle (square grid).
constexpr int NT_GRP = 8;
__host__ __device__ __forceinline__ int nt_tiles(int nmb, int nnb, bool lower) {
    return lower ? nmb * (nmb + 1) / 2 : nmb * nnb;
}
__host__ __device__ __forceinline__ void nt_tile_of(int t, int nmb, int nnb, bool lower, int& tm, int& tn) {
    if (!lower) {
        const int g = t / (NT_GRP * nnb), r0 = g * NT_GRP, in = t - g * NT_GRP * nnb;
        const int h = nmb - r0 < NT_GRP ? nmb - r0 : NT_GRP;
        tm = r0 + in % h;
        tn = in / h;
        return;
    }
    int r0 = 0;   // first row of the group: rows r0 .. r0 + h - 1 hold r0 + 1 .. r0 + h tiles
    for (;;) {
        const int h = nmb - r0 < NT_GRP ? nmb - r0 : NT_GRP;
        const int n = h * r0 + h * (h + 1) / 2;
        if (t < n || r0 + h >= nmb) {
            if (t < h * (r0 + 1)) {   // columns 0 .. r0: h tiles each
                tm = r0 + t % h;
                tn = t / h;
                return;
            }
            t -= h * (r0 + 1);
            int c = 1;                // columns r0 + c: the h - c rows from the diagonal on
            while (c < h - 1 && t >= h - c) {
                t -= h - c;
                c++;
            }
            tn = r0 + c;
            tm = tn + t;
            return;
        }
        t -= n;
        r0 += h;
    }
}

// Item -> band q, batch b and the tile's first row and column.
template <typename T, typename Out>
__device__ __forceinline__ void nt_item(const NtArgs<T>& g, int item, int& q, int& b, int& m0, int& n0) {
    const int nmb = (g.M + NT_BM - 1) / NT_BM, nnb = (g.N + NT_BN - 1) / NT_BN;
    const int tiles = nt_tiles(nmb, nnb, Out::lower);
    const int z = item / tiles;
    int tm, tn;
    nt_tile_of(item - z * tiles, nmb, nnb, Out::lower, tm, tn);
    q = z / g.nbat;
    b = z - q * g.nbat;
    m0 = tm * NT_BM;
    n0 = tn * NT_BN;
}

// One workgroup (4 waves, each 64 x 64 of the 128 x 128 tile) per work item, or
// (SPLIT) per work item and part of the K range, whose accumulators go to ws.  Operand rows go from global memory to LDS by the DMA
// loads of gfx950: a wave instruction fills 1 KB, eight rows of 128 bytes, lane
// L taking row L / 8 and the 16-byte chunk that the XOR swizzle puts in slot
// L % 8, so each row's 128 bytes are one coalesced segment and the fragment
// reads (16 rows, one chunk) touch every bank once.  A lane's 16-byte fragment read feeds 2 (FP64) or 4 (FP32) MFMAs: the
// four lane groups of an MFMA take k values of four different chunks, the same
// ones in both operands, which only permutes the sum over k within a step.
//
// Bound by the MFMA pipes: a wave's step is 64 MFMAs (4096 cycles in FP64) for
// 16 KB of fragment reads, and two workgroups per CU cover each other's waits
// (217 VGPRs, 64 KB of LDS each).  At 32^3 cells x 4000 modes FP64 stage 1 takes
// 132 ms per band (66.5 TFLOP/s; 179 ms with operands generated or staged through
// registers into k-major LDS and no overlap of LDS reads with MFMAs), stage 2
// 8.1 ms (64.6 TFLOP/s, 17.4 ms before); the library's dgemm reaches 72 on 8192^3.
template <typename T, typename Out, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void nt_gemm_kernel(NtArgs<T> g, Out O) {
    typedef typename NtMma<T>::acc_t acc_t;
    typedef typename NtMma<T>::vec_t vec_t;
    constexpr int NE = 16 / sizeof(T);
    extern __shared__ __attribute__((aligned(16))) char nt_lds[];
    // workgroups go to the eight XCDs round-robin: consecutive work items on one XCD
    const unsigned per = gridDim.x / 8;
    unsigned w = blockIdx.x;
    if (w < 8 * per) w = (w % 8) * per + w / 8;
    const int parts = SPLIT ? (int)gridDim.x / g.nsplit : 1, part = SPLIT ? (int)w / g.nsplit : 0;
    int q, b, m0, n0;
    nt_item<T, Out>(g, g.item0 + (int)w - part * g.nsplit, q, b, m0, n0);
    const T* A = g.A + (size_t)b * g.a_bs + (size_t)q * g.a_qs;
    const T* B = g.B + (size_t)q * g.b_qs + (size_t)((b + 1) >> 1) * g.b_bs;
    const int k0 = (int)((long long)part * g.ksteps / parts), k1 = (int)((long long)(part + 1) * g.ksteps / parts);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // this wave's eight DMA instructions: rows 8 (wave + 4 u) + lane / 8 of A, then of B
    const char *src[8];
    {
        const int r = lane >> 3, c = (lane & 7) ^ r;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int row = 8 * (wave + 4 * u) + r;
            src[u] = (const char*)(A + (size_t)min(m0 + row, g.M - 1) * g.lda) + 16 * c + (size_t)k0 * 128;
            src[4 + u] = (const char*)(B + (size_t)min(n0 + row, g.N - 1) * g.ldb) + 16 * c + (size_t)k0 * 128;
        }
    }
    auto issue = [&](int s) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
            __builtin_amdgcn_global_load_lds(src[u],
                                             (__attribute__((address_space(3))) void*)(nt_lds + s * NT_STAGE +
                                                                                      (u >> 2) * (NT_BM * 128) +
                                                                                      (wave + 4 * (u & 3)) * 1024),
                                             16, 0, 0);
            src[u] += 128;
        }
    };
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const int fr = lane & 15, slot = ((lane >> 4) ^ (fr & 7)) * 16;
    const int offA = (wm + fr) * 128 + slot, offB = NT_BM * 128 + (wn + fr) * 128 + slot;
    acc_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = acc_t{0, 0, 0, 0};
    vec_t a[2][4], bb[2][4];
    auto read = [&](const char* st, int h) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            a[h][i] = *(const vec_t*)(st + (offA ^ (64 * h)) + i * 2048);
            bb[h][i] = *(const vec_t*)(st + (offB ^ (64 * h)) + i * 2048);
        }
    };
    auto mul = [&](int h) {
#pragma unroll
        for (int e = 0; e < NE; e++)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = NtMma<T>::mma(a[h][i][e], bb[h][j][e], acc[i][j]);
    };
    // A step's first half of fragments is read from LDS under the previous step's
    // MFMAs.  The barrier sits between the halves: every wave has then read all it
    // needs of this stage, so the loads of step k + 2 go into it at once and have a
    // whole step to land.  The scheduling barriers keep the MFMAs on their side of
    // it (the compiler would otherwise wait for the loads first).
    issue(0);
    if (k0 + 1 < k1) issue(1);
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    read(nt_lds, 0);
    for (int k = k0; k < k1; k++) {
        const int cur = (k - k0) & 1;
        read(nt_lds + cur * NT_STAGE, 1);
        mul(0);
        __builtin_amdgcn_sched_barrier(0);
        if (k + 1 < k1) {
            __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (k + 2 < k1) issue(cur);
            read(nt_lds + (cur ^ 1) * NT_STAGE, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        mul(1);
    }
    if constexpr (SPLIT) {
        T* o = g.ws + (size_t)w * (NT_BM * NT_BN) + threadIdx.x;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) o[((i * 4 + j) * 4 + r) * 256] = acc[i][j][r];
    } else {
        auto* o = O.base(q, b);
        const bool in = O.inside(m0, n0, g.M);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm + i * 16 + acc_row<T>(lane, r), n = n0 + wn + fr;
                if (in) {
#pragma unroll
                    for (int j = 0; j < 4; j++) O.put_in(o, m, n + j * 16, acc[i][j][r]);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++) O.put(o, m, n + j * 16, g.M, acc[i][j][r]);
                }
            }
    }
}

// Split items: the parts of each accumulator added in order in FP64, then the epilogue.
// Four workgroups per item, one row of fragments each.
template <typename T, typename Out>
__global__ __launch_bounds__(256) void nt_fix_kernel(NtArgs<T> g, int parts, Out O) {
    int q, b, m0, n0;
    nt_item<T, Out>(g, g.item0 + (int)blockIdx.x, q, b, m0, n0);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = blockIdx.y;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const size_t stride = (size_t)g.nsplit * (NT_BM * NT_BN);
    const T* x = g.ws + (size_t)blockIdx.x * (NT_BM * NT_BN) + i * 16 * 256 + threadIdx.x;
    double v[16];
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = (double)x[e * 256];
    for (int p = 1; p < parts; p++)
#pragma unroll
        for (int e = 0; e < 16; e++) v[e] += (double)x[p * stride + e * 256];
    auto* o = O.base(q, b);
#pragma unroll
    for (int e = 0; e < 16; e++)
        O.put(o, m0 + wm + i * 16 + acc_row<T>(lane, e & 3), n0 + wn + (e >> 2) * 16 + (lane & 15), g.M, v[e]);
}

// Parts of the K range for the last `items` tiles of a launch (fewer than a
// round of two workgroups per CU), `ksteps` steps each; 1: do not split.  In
// steps (about 3.5 us): the unsplit items cost a whole round, about two thirds
// of one when no CU holds two (a lone workgroup does not hide its own waits);
// split, the parts' rounds, four steps of fill and drain each, and about four
// steps for the two more launches and the partial sums' traffic.  Measured at
// 1728 cells x 500 modes x 20 bands: stage 1 (1120 tiles) 1180 us unsplit, 953 +
// 104 + 12 us split; stage 2 (200 tiles) 253 us in one round, 204 + 26 us split.
inline int nt_split(int items, int ksteps, int cus) {
    const double slots = 2.0 * cus;
    if (items == 0) return 1;
    int best = 1;
    double cost = (items <= cus ? 0.67 : 1.0) * (ksteps + 4.0);
    for (int s = 2; s <= 32 && ksteps / s >= 4 && items * s <= 2 * slots; s++) {
        const double u = (double)items * s, full = std::floor(u / slots), rem = u - full * slots;
        const double rounds = full + (rem == 0 ? 0.0 : rem <= cus ? 0.67 : 1.0);
        const double c = rounds * ((double)ksteps / s + 4.0) + 4.0 + 0.004 * u;
        if (c < cost) {
            cost = c;
            best = s;
        }
    }
    return best;
}
// Workspace of the split launches, kept by its owner: at most two rounds of
// parts (128 MiB in FP64).
struct NtWork {
    void* p = nullptr;
    size_t cap = 0;
};

// All work items of g on ctx's stream: whole rounds of two workgroups per CU,
// then the rest, its K range split over the CUs when that pays and there is memory for the
// parts.
template <typename T, typename Out>
inline void launch_nt_gemm(opsec_ctx* ctx, NtWork& ws, NtArgs<T> g, const Out& O) {
    const int cus = std::max(1, ctx->num_cus);
    hipStream_t s = ctx->stream;
    const int nmb = (g.M + NT_BM - 1) / NT_BM, nnb = (g.N + NT_BN - 1) / NT_BN;
    const int total = nt_tiles(nmb, nnb, Out::lower) * g.nz, rest = total % (2 * cus);
    int parts = g.serial ? 1 : nt_split(rest, g.ksteps, cus);
    if (parts > 1 &&
        dev_try_realloc(&ws.p, &ws.cap, (size_t)rest * parts * NT_BM * NT_BN * sizeof(T)) != hipSuccess)
        parts = 1;
    const int whole = parts > 1 ? total - rest : total;
    g.item0 = 0;
    g.nsplit = 1;
    if (whole > 0) hipLaunchKernelGGL((nt_gemm_kernel<T, Out, false>), dim3(whole), dim3(256), NT_LDS, s, g, O);
    if (whole == total) return;
    g.ws = (T*)ws.p;
    g.item0 = whole;
    g.nsplit = rest;
    hipLaunchKernelGGL((nt_gemm_kernel<T, Out, true>), dim3(rest * parts), dim3(256), NT_LDS, s, g, O);
    hipLaunchKernelGGL((nt_fix_kernel<T, Out>), dim3(rest, 4), dim3(256), 0, s, g, parts, O);
}
// The same into rows that are an operand of the next product, in g's order.
template <typename T>
inline void launch_nt_gemm_rows(opsec_ctx* ctx, NtWork& ws, const NtArgs<T>& g, T* p, size_t ld, size_t q_stride, int nc,
                                int nw) {
    if constexpr (sizeof(T) == 4)
        if (g.serial) return launch_nt_gemm(ctx, ws, g, NtRows<T, true>{p, ld, 0, q_stride, nc, nw});
    launch_nt_gemm(ctx, ws, g, NtRows<T, false>{p, ld, 0, q_stride, nc, nw});
}

}  // namespace opsec
