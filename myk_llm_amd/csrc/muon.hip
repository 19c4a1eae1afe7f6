// Muon's batched Newton-Schulz iteration (ops/muon.py:218-268) as one call: Frobenius norms, the
// scaled (and, for tall matrices, transposed) bf16 copy, `steps` times three products (gemm.hip),
// and the way back to the caller's layout.
//   G = X X^T;  G2 = b G + c G G;  X' = a X + G2 X
// X lives as (batch, M, K) rows a multiple of 64 apart, zero up to the next multiple of 8, G and G2
// as (batch, M, M) likewise, so that every product reads its operands as they are: at 5 x 776 x 328 the padded
// copies before each product were 20 launches of the 45.
#include "common.h"
#include "kernels.h"

namespace mykfa {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxParts = 256;  // partial sums of squares per matrix
constexpr int kMaxBatch = 65535;  // matrices per launch, a grid dimension: more go in several runs
constexpr int kT = 64;          // transpose tile

int round8(int x) { return (x + 7) & ~7; }
int row_stride(int x) { return (x + 63) & ~63; }  // rows start 128-byte lines

// Sum over the workgroup in a fixed order; every thread gets it.
__device__ inline float block_sum(float x, float* red) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kThreads / 64; ++i) s += red[i];
    __syncthreads();
    return s;
}

// Partial sums of squares: part blockIdx.x of matrix blockIdx.y. HBM-bound (one read of x).
__global__ __launch_bounds__(kThreads) void square_sum_kernel(const uint16_t* x, int64_t n, float* part, int vec) {
    __shared__ float red[kThreads / 64];
    const uint16_t* p = x + blockIdx.y * n;
    const int64_t parts = gridDim.x, tid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    float s = 0.f;
    if (vec) {
        for (int64_t i = tid * 8; i < n; i += parts * kThreads * 8) {
            const s16x8 v = ld16(p + i);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float f = BF16::to_float((uint16_t)v[e]);
                s = fmaf(f, f, s);
            }
        }
    } else {
        for (int64_t i = tid; i < n; i += parts * kThreads) {
            const float f = BF16::to_float(p[i]);
            s = fmaf(f, f, s);
        }
    }
    s = block_sum(s, red);
    if (threadIdx.x == 0) part[blockIdx.y * parts + blockIdx.x] = s;
}

// The norm of matrix b, at least eps (a NaN stays one).
__device__ inline float matrix_norm(const float* part, int parts, int b, float eps, float* red) {
    const float s = block_sum((int)threadIdx.x < parts ? part[(int64_t)b * parts + threadIdx.x] : 0.f, red);
    const float norm = sqrtf(s);
    return norm < eps ? eps : norm;
}

__device__ inline s16x8 divide8(s16x8 v, float norm) {
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = BF16::to_float((uint16_t)v[e]) / norm;
    const u32x4 w = {BF16::pack2(f[0], f[1]), BF16::pack2(f[2], f[3]), BF16::pack2(f[4], f[5]), BF16::pack2(f[6], f[7])};
    return __builtin_bit_cast(s16x8, w);
}

// Up to 8 of the `left` elements from p on; the others zero.
__device__ inline s16x8 load_row8(const uint16_t* p, int left, bool vec) {
    if (vec && left >= 8) return ld16(p);
    s16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (e < left) v[e] = (short)p[e];
    return v;
}
__device__ inline void store_row8(uint16_t* p, s16x8 v, int left, bool vec) {
    if (vec && left >= 8) {
        st16(p, v);
        return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (e < left) p[e] = (uint16_t)v[e];
}

// A (rows, cols) matrix per blockIdx.z, row strides irs / ors, batch strides ibs / obs. part: divided by
// its norm. Output rows are written up to `owidth` columns, zeros past cols. One read, one write.
struct CopyArgs {
    const uint16_t* in;
    uint16_t* out;
    int64_t ibs, obs;
    int irs, ors, rows, cols, owidth;
    const float* part;
    int parts;
    float eps;
    int ivec, ovec;  // 16-byte rows on either side
};
__global__ __launch_bounds__(kThreads) void copy_kernel(CopyArgs a) {
    __shared__ float red[kThreads / 64];
    const int b = blockIdx.z;
    const float norm = a.part ? matrix_norm(a.part, a.parts, b, a.eps, red) : 1.f;
    const int cpr = (a.owidth + 7) / 8;
    const int64_t total = (int64_t)a.rows * cpr;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < total; i += (int64_t)gridDim.x * kThreads) {
        const int r = (int)(i / cpr), c = (int)(i % cpr) * 8;
        s16x8 v = load_row8(a.in + b * a.ibs + (int64_t)r * a.irs + c, a.cols - c, a.ivec);
        if (a.part) v = divide8(v, norm);
        store_row8(a.out + b * a.obs + (int64_t)r * a.ors + c, v, a.owidth - c, a.ovec);
    }
}
// The same transposed (output row c = input column c, its columns the input's rows), 64 x 64 tiles
// through LDS so that both sides move whole lines.
__global__ __launch_bounds__(kThreads) void transpose_kernel(CopyArgs a) {
    __shared__ float red[kThreads / 64];
    __shared__ __attribute__((aligned(16))) uint16_t tile[kT][kT + 8];  // [input column][input row]
    const int b = blockIdx.z, r0 = blockIdx.y * kT, c0 = blockIdx.x * kT;
    const float norm = a.part ? matrix_norm(a.part, a.parts, b, a.eps, red) : 1.f;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int r = 32 * q + threadIdx.x / 8, c = threadIdx.x % 8 * 8;
        s16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
        if (r0 + r < a.rows) v = load_row8(a.in + b * a.ibs + (int64_t)(r0 + r) * a.irs + c0 + c, a.cols - c0 - c, a.ivec);
        if (a.part) v = divide8(v, norm);
#pragma unroll
        for (int e = 0; e < 8; ++e) tile[c + e][r] = (uint16_t)v[e];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int c = 32 * q + threadIdx.x / 8, r = threadIdx.x % 8 * 8;
        if (c0 + c < a.cols && r0 + r < a.owidth)
            store_row8(a.out + b * a.obs + (int64_t)(c0 + c) * a.ors + r0 + r, *reinterpret_cast<const s16x8*>(&tile[c][r]),
                       a.owidth - r0 - r, a.ovec);
    }
}

__global__ __launch_bounds__(kThreads) void zero_kernel(s16x8* p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
        p[i] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
}

bool vec_rows(const void* p, int64_t bs, int64_t rs) {
    return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && bs % 8 == 0 && rs % 8 == 0;
}

hipError_t copy(CopyArgs a, int batch, bool transposed, hipStream_t s) {
    a.ivec = vec_rows(a.in, a.ibs, a.irs);
    a.ovec = vec_rows(a.out, a.obs, a.ors);
    if (transposed) {
        hipLaunchKernelGGL(transpose_kernel, dim3((a.cols + kT - 1) / kT, (a.owidth + kT - 1) / kT, batch), dim3(kThreads), 0,
                           s, a);
    } else {
        const long long chunks = (long long)a.rows * ((a.owidth + 7) / 8);
        const long long blocks = (chunks + kThreads * 4 - 1) / (kThreads * 4);  // four chunks a lane
        hipLaunchKernelGGL(copy_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096), 1, batch), dim3(kThreads), 0, s, a);
    }
    return hipGetLastError();
}

struct Sizes {
    int M, K;                    // X is (M, K)
    size_t x, g, part;           // bytes of one X buffer, of one G buffer, of the partial sums
};
Sizes sizes_of(const mykfa_newton_schulz_params& p) {  // of a run
    const int batch = p.batch < kMaxBatch ? p.batch : kMaxBatch;
    Sizes s;
    s.M = p.transposed ? p.cols : p.rows;
    s.K = p.transposed ? p.rows : p.cols;
    s.x = (size_t)batch * s.M * row_stride(s.K) * 2;
    s.g = (size_t)batch * s.M * row_stride(s.M) * 2;
    s.part = (size_t)batch * kMaxParts * sizeof(float);
    return s;
}
size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Up to kMaxBatch matrices.
hipError_t run(const mykfa_newton_schulz_params& p, void* ws, hipStream_t stream) {
    const Sizes z = sizes_of(p);
    const int M = z.M, K = z.K, M8 = round8(M), K8 = round8(K), Ms = row_stride(M), Ks = row_stride(K);
    char* w = static_cast<char*>(ws);
    uint16_t* xs[2] = {reinterpret_cast<uint16_t*>(w), reinterpret_cast<uint16_t*>(w + align256(z.x))};
    uint16_t* g = reinterpret_cast<uint16_t*>(w + 2 * align256(z.x));
    uint16_t* g2 = reinterpret_cast<uint16_t*>(w + 2 * align256(z.x) + align256(z.g));
    float* part = reinterpret_cast<float*>(w + 2 * align256(z.x) + 2 * align256(z.g));
    hipError_t e;

    const int64_t n = (int64_t)p.rows * p.cols;
    CopyArgs c{};
    c.in = static_cast<const uint16_t*>(p.x);
    c.out = xs[0];
    c.ibs = n; c.irs = p.cols;
    c.obs = (int64_t)M * Ks; c.ors = Ks;
    c.rows = p.rows; c.cols = p.cols; c.owidth = K8;
    c.eps = p.eps;
    if (!p.normalized) {
        // At least 8192 elements a part, 256 parts a matrix: the scaled copy sums them again.
        const int64_t want = (n + 8191) / 8192;
        c.part = part;
        c.parts = (int)(want < kMaxParts ? want : kMaxParts);
        hipLaunchKernelGGL(square_sum_kernel, dim3(c.parts, p.batch), dim3(kThreads), 0, stream, c.in, n, part,
                           vec_rows(c.in, n, 0) ? 1 : 0);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if ((e = copy(c, p.batch, p.transposed, stream)) != hipSuccess) return e;
    if (M8 != M) {  // G and G2 store no pads: their columns past M stay zero
        const int64_t chunks = (int64_t)((align256(z.g) * 2) / 16);
        hipLaunchKernelGGL(zero_kernel, dim3((unsigned)((chunks + 1023) / 1024 < 4096 ? (chunks + 1023) / 1024 : 4096)),
                           dim3(kThreads), 0, stream, reinterpret_cast<s16x8*>(g), chunks);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    // The last step's product goes straight to the caller's tensor where that has X's layout.
    const bool direct = !p.transposed && K8 == K && vec_rows(p.out, n, K);
    mykfa_gemm_params q{};
    q.batch = p.batch;
    q.c_dtype = MYKFA_BF16;
    const uint16_t* x = xs[0];
    for (int i = 0; i < p.steps; ++i) {
        const bool last = i + 1 == p.steps && direct;
        uint16_t* next = last ? static_cast<uint16_t*>(p.out) : xs[(i + 1) & 1];
        q.symmetric = 1;
        q.m = q.n = M;
        q.a = x; q.a_batch_stride = (int64_t)M * Ks; q.a_row_stride = Ks; q.k = K8;
        q.add = nullptr; q.alpha = 1.f; q.beta = 0.f;
        q.c = g; q.c_batch_stride = (int64_t)M * Ms; q.c_row_stride = Ms;
        if ((e = launch_gemm(q, nullptr, stream)) != hipSuccess) return e;
        q.a = g; q.a_batch_stride = (int64_t)M * Ms; q.a_row_stride = Ms; q.k = M8;
        q.add = g; q.add_batch_stride = (int64_t)M * Ms; q.add_row_stride = Ms;
        q.alpha = p.c; q.beta = p.b;
        q.c = g2;
        if ((e = launch_gemm(q, nullptr, stream)) != hipSuccess) return e;
        q.symmetric = 0;
        q.a = g2; q.m = M; q.n = K; q.k = M;
        q.b = x; q.b_batch_stride = (int64_t)M * Ks; q.b_row_stride = Ks;
        q.add = x; q.add_batch_stride = (int64_t)M * Ks; q.add_row_stride = Ks;
        q.alpha = 1.f; q.beta = p.a;
        q.c = next; q.c_batch_stride = (int64_t)M * (last ? K8 : Ks); q.c_row_stride = last ? K8 : Ks;
        if ((e = launch_gemm(q, nullptr, stream)) != hipSuccess) return e;
        x = next;
    }
    if (direct && p.steps > 0) return hipSuccess;
    CopyArgs o{};
    o.in = x;
    o.out = static_cast<uint16_t*>(p.out);
    o.ibs = (int64_t)M * Ks; o.irs = Ks;
    o.obs = n; o.ors = p.cols;
    o.rows = M; o.cols = K; o.owidth = p.transposed ? M : K;
    return copy(o, p.batch, p.transposed, stream);
}

}  // namespace

size_t newton_schulz_bytes(const mykfa_newton_schulz_params& p) {
    const Sizes s = sizes_of(p);
    return 2 * align256(s.x) + 2 * align256(s.g) + align256(s.part);
}

hipError_t launch_newton_schulz(const mykfa_newton_schulz_params& p, void* ws, hipStream_t stream) {
    for (int b = 0; b < p.batch; b += kMaxBatch) {
        mykfa_newton_schulz_params q = p;
        const int64_t at = (int64_t)b * p.rows * p.cols;
        q.x = static_cast<const uint16_t*>(p.x) + at;
        q.out = static_cast<uint16_t*>(p.out) + at;
        q.batch = p.batch - b < kMaxBatch ? p.batch - b : kMaxBatch;
        const hipError_t e = run(q, ws, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace mykfa
