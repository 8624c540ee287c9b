// qdequant.hip -- format kernels: dequantize, quantize, and the generic
// one-thread-per-output matmul used for shapes the tiled kernels reject.
#include "kernels.h"
#include "qcommon.h"

namespace lxq {

namespace {

// code k of a row, runtime bit width
__device__ __forceinline__ uint32_t row_code(const uint32_t* __restrict__ row, int k, int bits) {
    const uint32_t bit = (uint32_t)k * (uint32_t)bits, wi = bit >> 5, sh = bit & 31u;
    uint64_t pair = row[wi];
    if (sh + (uint32_t)bits > 32u) pair |= (uint64_t)row[wi + 1] << 32;
    return (uint32_t)(pair >> sh) & ((1u << bits) - 1u);
}

// Dequantizer.  Rows of codes, scales and outputs are each contiguous over the
// whole [N, K] matrix (K is a multiple of the group size), so chunk t = the CH
// codes CH t .. CH t + CH - 1 starts at bit CH t BITS of w_q, fills 16 bytes of
// the output (CH = 8 of 16-bit, 4 of f32 outputs) and lies in one group.  Lane
// = chunk: a wave reads contiguous codes and writes 1 KB.
// Bound by HBM, by the output above all (117 of 150 MB at N = 14336, K = 4096,
// 4-bit, f16); U chunks per lane, 256 apart, put U code and scale loads in
// flight before the first store.  One lane per code, a 64-bit division per
// code and 2-byte stores took 149 us at that size (1.0 TB/s), this 30.4 (5.0);
// f32 outputs (3-bit, group 32) as two 16-byte halves per lane, 32 bytes
// apart, 72 us, as one 60.7 (4.4).
template <int SB>
__device__ __forceinline__ float sb_at(const void* p, size_t i) {
    if constexpr (SB == DT_F32) return static_cast<const float*>(p)[i];
    else if constexpr (SB == DT_F16) return f16_to_f32(static_cast<const uint16_t*>(p)[i]);
    else return bf16_to_f32(static_cast<const uint16_t*>(p)[i]);
}

template <int BITS, int SB, int OT, int U>
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t* __restrict__ wq, const void* __restrict__ sc,
                                                      const void* __restrict__ bi, void* __restrict__ out,
                                                      size_t chunks, int gshift) {
    constexpr int CH = OT == DT_F32 ? 4 : 8;
    constexpr int CB = CH * BITS;  // bits of a chunk
    typedef uint32_t o4 __attribute__((ext_vector_type(4)));
    const size_t t0 = (size_t)blockIdx.x * (256 * U) + threadIdx.x;
    uint32_t lo[U], hi[U];
    float s[U], b[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const size_t t = t0 + 256 * u < chunks ? t0 + 256 * u : chunks - 1;
        // the chunk's bits in the low end of hi:lo; where they are not whole
        // words, from the two words they start in (up to 16 + 48 bits: the
        // second word may lie past w_q, in its readable tail)
        if constexpr (CB == 8) {
            lo[u] = reinterpret_cast<const uint8_t*>(wq)[t];
        } else if constexpr (CB == 16) {
            lo[u] = reinterpret_cast<const uint16_t*>(wq)[t];
        } else if constexpr (CB == 32) {
            lo[u] = wq[t];
        } else {
            const size_t bit = t * CB;
            const u32x2 v = *reinterpret_cast<const u32x2*>(wq + (bit >> 5));
            const uint32_t sh = (uint32_t)bit & 31u;
            lo[u] = CB == 64 ? v.x : __builtin_amdgcn_alignbit(v.y, v.x, sh);
            hi[u] = CB == 64 ? v.y : v.y >> sh;
        }
        const size_t g = t >> gshift;
        s[u] = sb_at<SB>(sc, g);
        b[u] = sb_at<SB>(bi, g);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const size_t t = t0 + 256 * u;
        if (t >= chunks) return;
        float v[CH];
#pragma unroll
        for (int i = 0; i < CH; i++) {
            constexpr uint32_t mask = (1u << BITS) - 1u;
            const int bit = i * BITS;
            const uint32_t q = bit + BITS <= 32 ? (lo[u] >> bit) & mask
                               : bit >= 32      ? (hi[u] >> (bit - 32)) & mask
                                                : __builtin_amdgcn_alignbit(hi[u], lo[u], bit) & mask;
            v[i] = fmaf(s[u], (float)q, b[u]);
        }
        o4* o = static_cast<o4*>(out) + t;
        if constexpr (OT == DT_F32) {
            typedef float f4 __attribute__((ext_vector_type(4)));
            *o = __builtin_bit_cast(o4, f4{v[0], v[1], v[2], v[3]});
        } else {
            *o = o4{pack2<OT>(v[0], v[1]), pack2<OT>(v[2], v[3]), pack2<OT>(v[4], v[5]), pack2<OT>(v[6], v[7])};
        }
    }
}

// Quantizer.  Lane t takes the 8 consecutive weights 8t .. 8t+7 of the
// row-major [N, K] matrix (one 16- or 32-byte load; a wave reads 512
// consecutive weights), so a group of GS weights spans GS/8 adjacent lanes
// and 8 codes of BITS bits are exactly BITS bytes at byte 8t*BITS/8 of the
// packed stream (rows are contiguous in both).  Per group, following the
// CPU quantizer's sequential scan (oracle/lux_cpu_quant.c, lux_cpu_quantize):
// mn/mx start at the group's first weight and take a later weight only if
// strictly smaller/larger, so a NaN first weight poisons the group and later
// NaNs are skipped, and ties keep the first occurrence.  The lanes of a group
// combine their partial results in index order (the lower segment wins
// ties); lanes other than the group's first start from +inf / -inf.
template <int WDT>
__device__ __forceinline__ void load8(const void* w, size_t e, float (&v)[8]) {
    if constexpr (WDT == DT_F32) {
        const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(w) + e);
        const float4 a = p[0], b = p[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
        const uint4 a = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(w) + e);
        const uint32_t d[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[2 * i] = WDT == DT_F16 ? f16_to_f32(d[i] & 0xffffu) : bf16_to_f32(d[i] & 0xffffu);
            v[2 * i + 1] = WDT == DT_F16 ? f16_to_f32(d[i] >> 16) : bf16_to_f32(d[i] >> 16);
        }
    }
}

template <int BITS, int WDT>
__global__ __launch_bounds__(256) void quantize_kernel(const void* __restrict__ w, uint32_t* __restrict__ wq,
                                                       void* __restrict__ sc, void* __restrict__ bi,
                                                       size_t chunks, int gsize, int sb_dt) {
    __shared__ __attribute__((aligned(16))) uint8_t pk[4][64 * 8];  // per wave: 64 lanes x BITS bytes
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t t0 = ((size_t)blockIdx.x * 4 + wave) * 64;  // first chunk of this wave
    const size_t t = t0 + lane;
    const bool act = t < chunks;
    const int L = gsize >> 3;    // lanes per group (4, 8 or 16; groups start at lane multiples of L)
    const int lig = lane & (L - 1);
    float v[8];
    if (act) {
        load8<WDT>(w, 8 * t, v);
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = 0.f;
    }
    float mn = lig == 0 ? v[0] : __builtin_inff(), mx = lig == 0 ? v[0] : -__builtin_inff();
#pragma unroll
    for (int i = 0; i < 8; i++) {
        mn = v[i] < mn ? v[i] : mn;
        mx = v[i] > mx ? v[i] : mx;
    }
    for (int d = 1; d < L; d <<= 1) {
        const float omn = __shfl_xor(mn, d), omx = __shfl_xor(mx, d);
        const bool up = lane & d;  // this lane holds the upper (later) segment
        const float lmn = up ? omn : mn, umn = up ? mn : omn;
        const float lmx = up ? omx : mx, umx = up ? mx : omx;
        mn = umn < lmn ? umn : lmn;
        mx = umx > lmx ? umx : lmx;
    }
    const float levels = (float)((1u << BITS) - 1u);
    // the codes are computed from the stored (rounded) scale and bias
    const float s = round_dt((mx - mn) / levels, sb_dt), b = round_dt(mn, sb_dt);
    if (act && lig == 0) {
        const size_t gi = 8 * t / (size_t)gsize;
        store_f(sc, gi, sb_dt, s);
        store_f(bi, gi, sb_dt, b);
    }
    uint64_t chunk = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        uint32_t q = 0;
        if (s != 0.0f) {
            float r = rintf((v[i] - b) / s);
            r = (r >= 0.0f) ? r : 0.0f;  // NaN -> 0
            r = r > levels ? levels : r;
            q = (uint32_t)r;
        }
        chunk |= (uint64_t)q << (i * BITS);
    }
    // the wave's packed bytes are contiguous: stage them in LDS, store whole dwords
#pragma unroll
    for (int y = 0; y < BITS; y++) pk[wave][lane * BITS + y] = (uint8_t)(chunk >> (8 * y));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // this wave's bytes [t0 BITS, min(t0 + 64, chunks) BITS): whole dwords, since
    // both ends are multiples of 4 (64 BITS, and N K BITS / 8 with K % 32 == 0)
    if (t0 < chunks) {
        const int nwords = (int)((chunks - t0 < 64) ? (chunks - t0) : 64) * BITS / 4;  // up to 16 BITS
        for (int i = lane; i < nwords; i += 64)
            wq[t0 * BITS / 4 + i] = reinterpret_cast<const uint32_t*>(pk[wave])[i];
    }
}

// y[m, n] = sum_k x * fmaf(s, q, b): fp32, ascending k, separate multiply and
// add (no contraction), the same order as the CPU oracle
__global__ __launch_bounds__(256) void qmm_generic_kernel(const void* __restrict__ x,
                                                          const uint32_t* __restrict__ wq,
                                                          const void* __restrict__ sc,
                                                          const void* __restrict__ bi,
                                                          void* __restrict__ y, int M, int K,
                                                          int N, int gsize, int bits, int x_dt,
                                                          int sb_dt, Epilogue ep) {
#pragma clang fp contract(off)
    const size_t total = (size_t)M * N;
    const int G = K / gsize, rw = (K * bits) >> 5;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (size_t)gridDim.x * blockDim.x) {
        const int n = (int)(i % N), m = (int)(i / N);
        const uint32_t* row = wq + (size_t)n * rw;
        float acc = 0.f;
        for (int k = 0; k < K; k++) {
            const size_t gi = (size_t)n * G + k / gsize;
            const float wv = fmaf(load_f(sc, gi, sb_dt), (float)row_code(row, k, bits),
                                  load_f(bi, gi, sb_dt));
            acc = acc + load_f(x, (size_t)m * K + k, x_dt) * wv;
        }
        store_out<true>(y, i, n, ep, acc);
    }
}

unsigned grid_for(size_t total) {
    size_t b = (total + 255) / 256;
    return (unsigned)(b < 65536 ? (b ? b : 1) : 65536);
}

}  // namespace

namespace {
// 4 chunks per lane where that still leaves every CU two blocks, else one
template <int BITS, int SB, int OT>
LuxStatus launch_dequant_t(const uint32_t* wq, const void* sc, const void* bi, void* out, size_t chunks, int gshift,
                           hipStream_t st) {
    if (chunks >= (size_t)512 * 1024) {
        hipLaunchKernelGGL((dequant_kernel<BITS, SB, OT, 4>), dim3((unsigned)((chunks + 1023) / 1024)), dim3(256), 0,
                           st, wq, sc, bi, out, chunks, gshift);
    } else {
        hipLaunchKernelGGL((dequant_kernel<BITS, SB, OT, 1>), dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, st,
                           wq, sc, bi, out, chunks, gshift);
    }
    return hipGetLastError() == hipSuccess ? LuxStatus::Ok : LuxStatus::Internal;
}
template <int BITS, int SB>
LuxStatus launch_dequant_o(const uint32_t* wq, const void* sc, const void* bi, void* out, size_t chunks, int gshift,
                           int out_dt, hipStream_t st) {
    switch (out_dt) {
    case DT_F32: return launch_dequant_t<BITS, SB, DT_F32>(wq, sc, bi, out, chunks, gshift, st);
    case DT_F16: return launch_dequant_t<BITS, SB, DT_F16>(wq, sc, bi, out, chunks, gshift, st);
    default: return launch_dequant_t<BITS, SB, DT_BF16>(wq, sc, bi, out, chunks, gshift, st);
    }
}
template <int BITS>
LuxStatus launch_dequant_b(const uint32_t* wq, const void* sc, const void* bi, void* out, size_t chunks, int gshift,
                           int sb_dt, int out_dt, hipStream_t st) {
    switch (sb_dt) {
    case DT_F32: return launch_dequant_o<BITS, DT_F32>(wq, sc, bi, out, chunks, gshift, out_dt, st);
    case DT_F16: return launch_dequant_o<BITS, DT_F16>(wq, sc, bi, out, chunks, gshift, out_dt, st);
    default: return launch_dequant_o<BITS, DT_BF16>(wq, sc, bi, out, chunks, gshift, out_dt, st);
    }
}
}  // namespace

LuxStatus launch_dequantize(const uint32_t* wq, const void* scales, const void* biases, void* out,
                            int N, int K, int group_size, int bits, int sb_dtype, int out_dtype,
                            hipStream_t st) {
    const int ch = out_dtype == DT_F32 ? 4 : 8;  // codes per chunk; group sizes are 32, 64 and 128, so K % 8 == 0
    const size_t chunks = (size_t)N * K / ch;
    if (chunks == 0) return LuxStatus::Ok;
    const int gshift = (group_size == 32 ? 5 : group_size == 64 ? 6 : 7) - (ch == 4 ? 2 : 3);  // chunks per group, log2
    switch (bits) {
    case 2: return launch_dequant_b<2>(wq, scales, biases, out, chunks, gshift, sb_dtype, out_dtype, st);
    case 3: return launch_dequant_b<3>(wq, scales, biases, out, chunks, gshift, sb_dtype, out_dtype, st);
    case 4: return launch_dequant_b<4>(wq, scales, biases, out, chunks, gshift, sb_dtype, out_dtype, st);
    case 5: return launch_dequant_b<5>(wq, scales, biases, out, chunks, gshift, sb_dtype, out_dtype, st);
    case 6: return launch_dequant_b<6>(wq, scales, biases, out, chunks, gshift, sb_dtype, out_dtype, st);
    case 8: return launch_dequant_b<8>(wq, scales, biases, out, chunks, gshift, sb_dtype, out_dtype, st);
    default: return LuxStatus::NotSupported;
    }
}

namespace {
template <int BITS, int WDT>
void launch_quantize_t(const void* w, uint32_t* wq, void* scales, void* biases, size_t chunks, int group_size,
                       int sb_dtype, hipStream_t st) {
    const size_t blocks = (chunks + 255) / 256;
    hipLaunchKernelGGL((quantize_kernel<BITS, WDT>), dim3((unsigned)blocks), dim3(256), 0, st, w, wq, scales, biases,
                       chunks, group_size, sb_dtype);
}
template <int WDT>
LuxStatus launch_quantize_w(const void* w, uint32_t* wq, void* sc, void* bi, size_t chunks, int gs, int bits,
                            int sb, hipStream_t st) {
    switch (bits) {
    case 2: launch_quantize_t<2, WDT>(w, wq, sc, bi, chunks, gs, sb, st); break;
    case 3: launch_quantize_t<3, WDT>(w, wq, sc, bi, chunks, gs, sb, st); break;
    case 4: launch_quantize_t<4, WDT>(w, wq, sc, bi, chunks, gs, sb, st); break;
    case 5: launch_quantize_t<5, WDT>(w, wq, sc, bi, chunks, gs, sb, st); break;
    case 6: launch_quantize_t<6, WDT>(w, wq, sc, bi, chunks, gs, sb, st); break;
    case 8: launch_quantize_t<8, WDT>(w, wq, sc, bi, chunks, gs, sb, st); break;
    default: return LuxStatus::NotSupported;
    }
    return hipGetLastError() == hipSuccess ? LuxStatus::Ok : LuxStatus::Internal;
}
}  // namespace

LuxStatus launch_quantize(const void* w, uint32_t* wq, void* scales, void* biases, int N, int K,
                          int group_size, int bits, int w_dtype, int sb_dtype, hipStream_t st) {
    const size_t chunks = (size_t)N * K / 8;  // 8 weights per lane; group sizes are 32, 64, 128
    if (chunks == 0) return LuxStatus::Ok;
    if (group_size != 32 && group_size != 64 && group_size != 128) return LuxStatus::NotSupported;
    // one block per 256 lanes: the grid's x dimension holds up to 2^31 - 1 blocks
    if ((chunks + 255) / 256 >= (1ull << 31)) return LuxStatus::NotSupported;
    switch (w_dtype) {
    case DT_F32: return launch_quantize_w<DT_F32>(w, wq, scales, biases, chunks, group_size, bits, sb_dtype, st);
    case DT_F16: return launch_quantize_w<DT_F16>(w, wq, scales, biases, chunks, group_size, bits, sb_dtype, st);
    default: return launch_quantize_w<DT_BF16>(w, wq, scales, biases, chunks, group_size, bits, sb_dtype, st);
    }
}

LuxStatus launch_qmm_generic(const QmmArgs& a, hipStream_t st) {
    const size_t total = (size_t)a.M * a.N;
    if (total == 0) return LuxStatus::Ok;
    if (planned(a, "qmm_generic_kernel")) return LuxStatus::Ok;
    hipLaunchKernelGGL(qmm_generic_kernel, dim3(grid_for(total)), dim3(256), 0, st, a.x, a.wq,
                       a.scales, a.biases, a.y, a.M, a.K, a.N, a.group_size, a.bits, a.x_dtype,
                       a.sb_dtype, a.epi());
    return hipGetLastError() == hipSuccess ? LuxStatus::Ok : LuxStatus::Internal;
}

}  // namespace lxq
