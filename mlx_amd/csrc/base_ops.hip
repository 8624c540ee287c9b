// base_ops.hip -- the plugin ABI's f32 tensor ops on the GPU: elementwise
// add / sub / mul / div, matmul and transpose, with the reference CPU
// backend's semantics (src/cpu_backend.cpp:185-266): IEEE fp32 per element,
// and for matmul C[M,N] = A[M,K] . B[K,N] (row-major) with every output
// summed in ascending k as a separate multiply and add, so the results are
// bit-identical to the CPU backend's.
#include <algorithm>

#include "kernels.h"

namespace lxq {
namespace {

enum : int { EW_ADD = 0, EW_SUB = 1, EW_MUL = 2, EW_DIV = 3 };

// 4 elements per thread (a 16-byte load of each operand), grid-stride
template <int OP>
__global__ __launch_bounds__(256) void ew_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                 float* __restrict__ o, size_t n) {
#pragma clang fp contract(off)
    const size_t n4 = n / 4;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
        const float4 x = reinterpret_cast<const float4*>(a)[i], y = reinterpret_cast<const float4*>(b)[i];
        float4 r;
        if constexpr (OP == EW_ADD) r = make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w);
        else if constexpr (OP == EW_SUB) r = make_float4(x.x - y.x, x.y - y.y, x.z - y.z, x.w - y.w);
        else if constexpr (OP == EW_MUL) r = make_float4(x.x * y.x, x.y * y.y, x.z * y.z, x.w * y.w);
        else r = make_float4(x.x / y.x, x.y / y.y, x.z / y.z, x.w / y.w);
        reinterpret_cast<float4*>(o)[i] = r;
    }
    // tail (n % 4 elements) by the first threads
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n - 4 * n4) {
        const size_t i = 4 * n4 + t;
        float r;
        if constexpr (OP == EW_ADD) r = a[i] + b[i];
        else if constexpr (OP == EW_SUB) r = a[i] - b[i];
        else if constexpr (OP == EW_MUL) r = a[i] * b[i];
        else r = a[i] / b[i];
        o[i] = r;
    }
}

// Tiled matmul: a block of 256 threads computes a TM x TN tile of C, each
// thread an RM x RN micro-tile of adjacent rows and columns; A and B advance
// through two LDS stages TK k at a time, the next stage's global loads in
// registers meanwhile (one barrier per stage).  Each output's sum still runs
// k = 0, 1, 2, ... with one rounding per multiply and per add (no
// contraction), the CPU backend's order, so K is never split.
//
// KM = 1 (wide micro-tiles): both operands k-major in LDS, one 16-byte read
// per 4 rows or columns and k.  KM = 4 (RM, RN <= 2): row-major, one 16-byte
// read per row or column and 4 k.
//
// Bound by VALU issue (32-bit multiply and add, packed forms excluded): 55
// TFLOP/s at 2048^3 and 40 to 43 at 1000 x 2000 x 3000 (281 to 298 us by box),
// where one multiply-add pair per lane and 4 clocks would be 39 and two 78.
// 4 x 4 tiles read from LDS word by word, k by k, took 474 us there.
template <int TM_, int TN_, int RM_, int RN_, int TK_, int KM_>
struct MmTile {
    static constexpr int TM = TM_, TN = TN_, RM = RM_, RN = RN_, TK = TK_, KM = KM_;
    static constexpr int kAV = TM * TK / 1024, kBV = TK * TN / 1024;  // 16-byte loads per thread and stage
    // LDS floats per stage: [k][m] and [k][n], or [m][k] and [n][k] (rows 16
    // bytes apart modulo the banks)
    static constexpr int kAS = KM == 1 ? TM + 4 : TK + 4, kBS = KM == 1 ? TN : TK + 4;
    static constexpr int kA = (KM == 1 ? TK : TM) * kAS, kB = (KM == 1 ? TK : TN) * kBS;
    static_assert(TM / RM * (TN / RN) == 256 && kAV >= 1 && kBV >= 1, "256 threads, whole loads");
    static_assert(2 * 4 * (kA + kB) <= 64 * 1024, "static LDS");
};

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // rows of A and B are dword-aligned only
typedef float f4a __attribute__((ext_vector_type(4)));

template <class T>
__global__ __launch_bounds__(256) void matmul_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                     float* __restrict__ C, int M, int K, int N) {
#pragma clang fp contract(off)
    constexpr int TM = T::TM, TN = T::TN, RM = T::RM, RN = T::RN, TK = T::TK, KM = T::KM;
    __shared__ __attribute__((aligned(16))) float As[2][T::kA];
    __shared__ __attribute__((aligned(16))) float Bs[2][T::kB];
    const int tid = threadIdx.x;
    const int tx = tid % (TN / RN), ty = tid / (TN / RN);
    const int ntiles = (N + TN - 1) / TN;
    const int m0 = (int)(blockIdx.x / (unsigned)ntiles) * TM, n0 = (int)(blockIdx.x % (unsigned)ntiles) * TN;
    // the loads of a stage: 4 k of a row of A, 4 columns of a row of B.  Rows
    // past M and K re-read the last one; a load that runs past its row's end
    // reads the next row, or up to 12 bytes of the buffer's readable tail:
    // such values feed padded k, which never enter a sum, or outputs that
    // are not stored
    const float* ap[T::kAV];
    int am[T::kAV], ak[T::kAV], bk[T::kBV], bn[T::kBV];
#pragma unroll
    for (int r = 0; r < T::kAV; r++) {
        const int e = tid + 256 * r;
        am[r] = e / (TK / 4);
        ak[r] = e % (TK / 4) * 4;
        ap[r] = A + (size_t)(m0 + am[r] < M ? m0 + am[r] : M - 1) * K;
    }
#pragma unroll
    for (int r = 0; r < T::kBV; r++) {
        const int e = tid + 256 * r;
        bk[r] = e / (TN / 4);
        bn[r] = e % (TN / 4) * 4;
    }
    f4u av[T::kAV], bv[T::kBV];
    auto load = [&](int k0) {
#pragma unroll
        for (int r = 0; r < T::kAV; r++) av[r] = *reinterpret_cast<const f4u*>(ap[r] + (k0 + ak[r] < K ? k0 + ak[r] : K - 1));
#pragma unroll
        for (int r = 0; r < T::kBV; r++) {
            const int k = k0 + bk[r] < K ? k0 + bk[r] : K - 1, n = n0 + bn[r] < N ? n0 + bn[r] : N - 1;
            bv[r] = *reinterpret_cast<const f4u*>(B + (size_t)k * N + n);
        }
    };
    auto store = [&](int st) {
#pragma unroll
        for (int r = 0; r < T::kAV; r++) {
            if constexpr (KM == 1) {
#pragma unroll
                for (int i = 0; i < 4; i++) As[st][(ak[r] + i) * T::kAS + am[r]] = av[r][i];
            } else {
                *reinterpret_cast<f4a*>(&As[st][am[r] * T::kAS + ak[r]]) = av[r];
            }
        }
#pragma unroll
        for (int r = 0; r < T::kBV; r++) {
            if constexpr (KM == 1) {
                *reinterpret_cast<f4a*>(&Bs[st][bk[r] * T::kBS + bn[r]]) = bv[r];
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) Bs[st][(bn[r] + i) * T::kBS + bk[r]] = bv[r][i];
            }
        }
    };
    float acc[RM][RN] = {};
    // operands of steps k .. k + KM - 1, and their multiply-adds (nk of them)
    struct Ops {
        float a[RM][KM], b[RN][KM];
    };
    auto read = [&](int st, int k, Ops& o) {
        if constexpr (KM == 1) {
#pragma unroll
            for (int i = 0; i < RM; i++) o.a[i][0] = As[st][k * T::kAS + ty * RM + i];
#pragma unroll
            for (int j = 0; j < RN; j++) o.b[j][0] = Bs[st][k * T::kBS + tx * RN + j];
        } else {
#pragma unroll
            for (int i = 0; i < RM; i++) {
                const f4a v = *reinterpret_cast<const f4a*>(&As[st][(ty * RM + i) * T::kAS + k]);
#pragma unroll
                for (int e = 0; e < KM; e++) o.a[i][e] = v[e];
            }
#pragma unroll
            for (int j = 0; j < RN; j++) {
                const f4a v = *reinterpret_cast<const f4a*>(&Bs[st][(tx * RN + j) * T::kBS + k]);
#pragma unroll
                for (int e = 0; e < KM; e++) o.b[j][e] = v[e];
            }
        }
    };
    auto mac = [&](const Ops& o, int nk) {
#pragma unroll
        for (int e = 0; e < KM; e++) {
            if (e >= nk) break;
#pragma unroll
            for (int i = 0; i < RM; i++)
#pragma unroll
                for (int j = 0; j < RN; j++) acc[i][j] = acc[i][j] + o.a[i][e] * o.b[j][e];
        }
    };
    load(0);
    store(0);
    __syncthreads();
    int st = 0;
    for (int k0 = 0; k0 < K; k0 += TK, st ^= 1) {
        const bool more = k0 + TK < K;
        if (more) load(k0 + TK);
        if (k0 + TK <= K) {
            // LDS reads run PD batches ahead of their use
            constexpr int PD = 2, NB = TK / KM;
            Ops o[PD + 1];
#pragma unroll
            for (int k = 0; k < PD; k++) read(st, k * KM, o[k]);
#pragma unroll
            for (int k = 0; k < NB; k++) {
                if (k + PD < NB) read(st, (k + PD) * KM, o[(k + PD) % (PD + 1)]);
                mac(o[k % (PD + 1)], KM);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            for (int k = 0; k < K - k0; k += KM) {
                Ops o;
                read(st, k, o);
                mac(o, K - k0 - k);
            }
        }
        if (more) store(st ^ 1);
        __syncthreads();
    }
    // a row of the micro-tile in one store (dword-aligned, as rows of any N
    // are): value by value, lanes RN columns apart, M = 1429, K = 2, N = 4755
    // took 15.4 us, so 9.4; M = 1930, K = 15, N = 4674 22.9 and 15.6
    typedef float fr __attribute__((ext_vector_type(RN), aligned(4)));
    const int n = n0 + tx * RN;
#pragma unroll
    for (int i = 0; i < RM; i++) {
        const int m = m0 + ty * RM + i;
        if (m >= M) break;
        float* c = C + (size_t)m * N + n;
        if (n + RN <= N) {
            fr v;
#pragma unroll
            for (int j = 0; j < RN; j++) v[j] = acc[i][j];
            *reinterpret_cast<fr*>(c) = v;
        } else {
#pragma unroll
            for (int j = 0; j < RN - 1; j++)
                if (n + j < N) c[j] = acc[i][j];
        }
    }
}

// out[c][r] = in[r][c] through a 32 x 33 LDS tile (conflict-free both ways)
__global__ __launch_bounds__(256) void transpose_kernel(const float* __restrict__ in, float* __restrict__ out,
                                                        int rows, int cols) {
    __shared__ float t[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;  // 32 x 8 threads
    for (int i = ty; i < 32; i += 8) {
        const int r = r0 + i, c = c0 + tx;
        if (r < rows && c < cols) t[i][tx] = in[(size_t)r * cols + c];
    }
    __syncthreads();
    for (int i = ty; i < 32; i += 8) {
        const int c = c0 + i, r = r0 + tx;
        if (c < cols && r < rows) out[(size_t)c * rows + r] = t[tx][i];
    }
}

}  // namespace

LuxStatus launch_elementwise(int op, const float* a, const float* b, float* o, size_t n, hipStream_t st) {
    if (n == 0) return LuxStatus::Ok;
    size_t blocks = (n / 4 + 255) / 256;
    blocks = blocks < 1 ? 1 : blocks > 65536 ? 65536 : blocks;
    switch (op) {
    case EW_ADD: hipLaunchKernelGGL(ew_kernel<EW_ADD>, dim3((unsigned)blocks), dim3(256), 0, st, a, b, o, n); break;
    case EW_SUB: hipLaunchKernelGGL(ew_kernel<EW_SUB>, dim3((unsigned)blocks), dim3(256), 0, st, a, b, o, n); break;
    case EW_MUL: hipLaunchKernelGGL(ew_kernel<EW_MUL>, dim3((unsigned)blocks), dim3(256), 0, st, a, b, o, n); break;
    case EW_DIV: hipLaunchKernelGGL(ew_kernel<EW_DIV>, dim3((unsigned)blocks), dim3(256), 0, st, a, b, o, n); break;
    default: return LuxStatus::Invalid;
    }
    return hipGetLastError() == hipSuccess ? LuxStatus::Ok : LuxStatus::Internal;
}

namespace {
template <class T>
LuxStatus launch_mm(const float* a, const float* b, float* c, int M, int K, int N, hipStream_t st) {
    const size_t blocks = (size_t)((M + T::TM - 1) / T::TM) * (size_t)((N + T::TN - 1) / T::TN);
    if (blocks >= (1ull << 31)) return LuxStatus::NotSupported;
    hipLaunchKernelGGL(matmul_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, st, a, b, c, M, K, N);
    return hipGetLastError() == hipSuccess ? LuxStatus::Ok : LuxStatus::Internal;
}

// ns per k of a tile's launch: a block per CU costs `alone` however few the
// blocks (one wave per SIMD issues at half rate), more of them `round` per
// 256 blocks.  Measured at K = 1000, us per launch, tile against the next:
// M x N = 2000 x 4000 315 (128 x 64) against 325 and 352; 1000 x 3000 133
// (64 x 64) against 143 and 137; 1500 x 1500 113 (32 x 64) against 133 and
// 127; 500 x 1000 32 (32 x 32) against 48 and 42; 20 x 4000 14.4 (16 x 16)
// against 25 and 78 (64 x 64).
struct MmCost {
    int tm, tn, alone, round;
};
constexpr MmCost kMmCost[] = {
    {128, 64, 145, 79}, {64, 64, 80, 40}, {32, 64, 47, 23}, {32, 32, 25, 15}, {16, 16, 13, 6}};

int mm_tile(int M, int N) {
    int best = 0;
    size_t least = ~(size_t)0;
    for (int v = 0; v < 5; v++) {
        const MmCost& t = kMmCost[v];
        const size_t blocks = (size_t)((M + t.tm - 1) / t.tm) * (size_t)((N + t.tn - 1) / t.tn);
        const size_t ns = std::max<size_t>((size_t)t.alone, (blocks + 255) / 256 * (size_t)t.round);
        if (ns < least) { least = ns; best = v; }
    }
    return best;
}
}  // namespace

LuxStatus launch_matmul_f32(const float* a, const float* b, float* c, int M, int K, int N, hipStream_t st) {
    if (M == 0 || N == 0) return LuxStatus::Ok;
    if (K == 0) return hipMemsetAsync(c, 0, (size_t)M * N * 4, st) == hipSuccess ? LuxStatus::Ok : LuxStatus::Internal;
    if (M > 64 * 65535) return LuxStatus::NotSupported;
    switch (mm_tile(M, N)) {
    case 0: return launch_mm<MmTile<128, 64, 8, 4, 16, 1>>(a, b, c, M, K, N, st);
    case 1: return launch_mm<MmTile<64, 64, 4, 4, 32, 1>>(a, b, c, M, K, N, st);
    case 2: return launch_mm<MmTile<32, 64, 2, 4, 32, 1>>(a, b, c, M, K, N, st);
    case 3: return launch_mm<MmTile<32, 32, 2, 2, 64, 4>>(a, b, c, M, K, N, st);
    default: return launch_mm<MmTile<16, 16, 1, 1, 64, 4>>(a, b, c, M, K, N, st);
    }
}

LuxStatus launch_transpose_f32(const float* in, float* out, int rows, int cols, hipStream_t st) {
    if (rows == 0 || cols == 0) return LuxStatus::Ok;
    const dim3 grid((cols + 31) / 32, (rows + 31) / 32);
    if (grid.y > 65535) return LuxStatus::NotSupported;
    hipLaunchKernelGGL(transpose_kernel, grid, dim3(256), 0, st, in, out, rows, cols);
    return hipGetLastError() == hipSuccess ? LuxStatus::Ok : LuxStatus::Internal;
}

}  // namespace lxq
