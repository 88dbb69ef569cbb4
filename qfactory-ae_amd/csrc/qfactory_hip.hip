// libqfactory_hip.so: device-side repacking and memory-system calibration kernels for gfx950.
// Entry points and their contracts are declared in include/qfactory_hip.h.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <stdint.h>

#include "qfactory_hip.h"
#include "qfactory_hip_ext.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

int fail(const char* fn, const char* why) {
    fprintf(stderr, "%s: %s\n", fn, why);
    return 1;
}

int launched(const char* fn) {
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        fprintf(stderr, "%s: launch failed: %s\n", fn, hipGetErrorString(err));
        return 2;
    }
    return 0;
}

// ---------------------------------------------------------------------------------------------
// Weight repack, bound by memory: four bytes are read per field.  A block takes 128 columns n (64 by the rule of launch_layer)
// and 32 main-plane words of K (32 threads x 4 columns side by side, 16 units of K): a thread reads 16 bytes of every k of its
// unit -- 512 contiguous bytes per k and 32 threads -- builds four columns' words in registers, and the words change their orientation
// through LDS, so that a row of the output is written 128 bytes at a time.  (A 4-byte word per thread straight to its row left
// 32-byte pieces: 22016 x 4096 at 4 bits 102 us = 4.0 TB/s.  Through LDS by columns of a block, 22016 x 4096 / 4096 x 4096 / 8192 x
// 28672 at 4 bits: 32 columns 81 / 16.7 / 210 us, 64 73 / 15.1 / 190, 128 with 256 threads 71 / 14.1 / 183, 128 with 512 70.6 / 13.8 /
// 178 = 5.8 TB/s, 256 71 / 18.6 / 188.)  Both planes of the 3-bit layout come out of one read of the fields.
// Position j of a word holds element (j < P/2 ? 2j : 2(j - P/2) + 1) of its P = 32/b elements
// (identity for 8-bit): evens in the low half-word, odds in the high half-word.  The 1-bit plane
// of the 3-bit layout has its own order (hi_plane_pos): every high bit sits where one shift of
// the word drops it directly above the element's field in the 2-bit plane.
// Fields outside [0, 2^b) are counted by the same read: any bit above the field (a negative number has them all) is
// collected per thread, and a wave that saw one sets `bad`.
// ---------------------------------------------------------------------------------------------
__host__ __device__ constexpr int hi_plane_pos(int e) {
    const int r = e / 16, ep = e % 16, i = ep / 2, h = ep % 2, p = i % 4, upper = i / 4;
    return ((p % 2 == 0) ? 2 * p + 2 : 2 * p - 2) + 8 * upper + r + 16 * h;
}
// bit position of element e inside its word of a plane of B-bit fields
template <int B>
__host__ __device__ constexpr int field_bit(int e) {
    return B == 8 ? 8 * e : B == 1 ? hi_plane_pos(e) : B * (e / 2 + (e % 2) * (16 / B));
}

// the word may be host memory: a plain store at system scope
__device__ __forceinline__ void report(uint32_t* bad) {
    __hip_atomic_store(bad, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int NBITS_, int THREADS_>
struct PackCfg {
    static constexpr int NBITS = NBITS_, THREADS = THREADS_;
    static constexpr int B = NBITS == 3 ? 2 : NBITS;           // field width of the main plane
    static constexpr int P = 32 / B;                           // elements per main-plane word
    static constexpr int UNIT = NBITS == 3 ? 32 : (P < 8 ? 8 : P);      // elements of K per thread and pass
    static constexpr int UW = UNIT / P;                        // main-plane words per unit
    static constexpr int WORDS = 32;                           // main-plane words of a block
    static constexpr int COLS = THREADS / 4;              // its columns: sixteen units of K side by side
    static constexpr int PASSES = WORDS / UW / 16;
    static constexpr int KB = WORDS * P;                       // elements of K of a block
    static constexpr int HI = NBITS == 3 ? WORDS / 2 : 0;      // 1-bit-plane words of a block
    static constexpr int PITCH = WORDS + HI + 1;               // odd: the transposed accesses spread over the banks
};

// VEC: N a multiple of four and 16-byte aligned rows, four columns per load; otherwise single words
template <class C, bool VEC>
__device__ __forceinline__ void pack_weight_tile(int64_t bx, int64_t by, const int32_t* __restrict__ weight, uint32_t* __restrict__ out,
                                                 int64_t K, int64_t N, uint32_t* __restrict__ bad) {
    constexpr int NBITS = C::NBITS;
    __shared__ uint32_t tile[C::COLS][C::PITCH];
    const int tx = threadIdx.x % (C::COLS / 4), ty = threadIdx.x / (C::COLS / 4);
    const int64_t n0 = bx * C::COLS, n = n0 + 4 * tx;
    const int64_t k_blk = by * C::KB;
    constexpr uint32_t MASK = (1u << NBITS) - 1u;
    uint32_t seen = 0;
#pragma unroll
    for (int pass = 0; pass < C::PASSES; pass++) {
        const int unit = pass * 16 + ty;
        const int64_t k0 = k_blk + (int64_t)unit * C::UNIT;
        uint32_t word[4][C::UW] = {}, high[4] = {};
        if (k0 < K && n < N) {                                  // K is a multiple of 32, hence of the unit
            u32x4 v[C::UNIT];
#pragma unroll
            for (int e = 0; e < C::UNIT; e++) {
                const uint32_t* src = reinterpret_cast<const uint32_t*>(weight) + (k0 + e) * N + n;
                if constexpr (VEC) {
                    v[e] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src));
                } else {
#pragma unroll
                    for (int c = 0; c < 4; c++) v[e][c] = n + c < N ? src[c] : 0u;
                }
            }
#pragma unroll
            for (int e = 0; e < C::UNIT; e++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    seen |= v[e][c];
                    word[c][e / C::P] |= (v[e][c] & MASK & ((1u << C::B) - 1u)) << field_bit<C::B>(e % C::P);
                    if constexpr (NBITS == 3) high[c] |= ((v[e][c] >> 2) & 1u) << field_bit<1>(e);
                }
        }
#pragma unroll
        for (int c = 0; c < 4; c++) {
#pragma unroll
            for (int w = 0; w < C::UW; w++) tile[4 * tx + c][unit * C::UW + w] = word[c][w];
            if constexpr (NBITS == 3) tile[4 * tx + c][C::WORDS + unit] = high[c];
        }
    }
    if (bad != nullptr && __any((seen & ~MASK) != 0) && (threadIdx.x & 63) == 0) report(bad);
    __syncthreads();
    const int64_t row_words = K * NBITS / 32;
    const int64_t w0 = by * C::WORDS;
    for (int i = threadIdx.x; i < C::COLS * C::WORDS; i += C::THREADS) {
        const int r = i / C::WORDS, w = i % C::WORDS;
        if (n0 + r < N && w0 + w < K / C::P) out[(n0 + r) * row_words + w0 + w] = tile[r][w];
    }
    if constexpr (NBITS == 3) {                                 // the 1-bit plane behind the row's 2-bit plane
        const int64_t h0 = by * C::HI;
        for (int i = threadIdx.x; i < C::COLS * C::HI; i += C::THREADS) {
            const int r = i / C::HI, w = i % C::HI;
            if (n0 + r < N && h0 + w < K / 32) out[(n0 + r) * row_words + K / 16 + h0 + w] = tile[r][C::WORDS + w];
        }
    }
}

template <int THREADS>
__device__ __forceinline__ void pack_zero_tile(int64_t block, const int32_t* __restrict__ zero, uint8_t* __restrict__ out,
                                               int64_t G, int64_t N, int nbits, int fb, uint32_t* __restrict__ bad) {
    const int p8 = 8 / fb;
    const int64_t row_bytes = G / p8;
    const int64_t idx = block * THREADS + threadIdx.x;      // over N * row_bytes, n fastest
    if (idx >= N * row_bytes) return;
    const int64_t n = idx % N, byte = idx / N;
    const int32_t maxv = (1 << nbits) - 1;
    uint32_t v = 0, seen = 0;
    for (int i = 0; i < p8; i++) {
        int32_t z = zero[(byte * p8 + i) * N + n];
        seen |= (uint32_t)z;
        z = z == 0x7fffffff ? z : z + 1;
        z = z > maxv ? maxv : z;
        v |= (uint32_t)z << (i * fb);
    }
    out[n * row_bytes + byte] = (uint8_t)v;
    if (bad != nullptr && (seen & ~(uint32_t)maxv) != 0) report(bad);
}

template <int THREADS>
__device__ __forceinline__ void transpose_u16_tile(int64_t bx, int64_t by, const uint16_t* __restrict__ in, uint16_t* __restrict__ out,
                                                   int64_t G, int64_t N) {
    __shared__ uint16_t tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;           // 32 x THREADS / 32
    const int64_t n0 = bx * 32, g0 = by * 32;
    for (int r = ty; r < 32; r += THREADS / 32)
        if (g0 + r < G && n0 + tx < N) tile[r][tx] = in[(g0 + r) * N + n0 + tx];
    __syncthreads();
    for (int r = ty; r < 32; r += THREADS / 32)
        if (n0 + r < N && g0 + tx < G) out[(n0 + r) * G + g0 + tx] = tile[tx][r];
}

// The three tensors of a layer in one launch: the scale and zero-point blocks come first and run under the weight's (as
// launches of their own behind it they took 5 and 6 us on 4096 x 22016, almost all of it latency).  Any of the three may
// have no blocks.
struct PackJob {
    const int32_t* weight; uint32_t* w_out;
    const uint16_t* scale; uint16_t* s_out;
    const int32_t* zero; uint8_t* z_out;
    int64_t K, N, G;
    int nbits, fb;
    uint32_t* bad;
    unsigned scale_blocks, zero_blocks;
};

template <class C, bool VEC>
__global__ __launch_bounds__(C::THREADS) void pack_layer_kernel(PackJob j) {
    unsigned b = blockIdx.x;
    if (b < j.scale_blocks) {
        const unsigned columns = (unsigned)((j.N + 31) / 32);
        transpose_u16_tile<C::THREADS>(b % columns, b / columns, j.scale, j.s_out, j.G, j.N);
        return;
    }
    b -= j.scale_blocks;
    if (b < j.zero_blocks) {
        pack_zero_tile<C::THREADS>(b, j.zero, j.z_out, j.G, j.N, j.nbits, j.fb, j.bad);
        return;
    }
    b -= j.zero_blocks;
    const unsigned columns = (unsigned)((j.N + C::COLS - 1) / C::COLS);
    pack_weight_tile<C, VEC>(b % columns, b / columns, j.weight, j.w_out, j.K, j.N, j.bad);
}

template <class C>
int64_t weight_blocks(const PackJob& j) {
    return j.weight ? (j.N + C::COLS - 1) / C::COLS * ((j.K + C::KB - 1) / C::KB) : 0;
}

template <class C>
int launch_blocks(const char* fn, PackJob j, bool vec, hipStream_t stream) {
    const int64_t scale_blocks = j.scale ? (j.N + 31) / 32 * ((j.G + 31) / 32) : 0;
    const int64_t zero_blocks = j.zero ? (j.N * (j.G / (8 / j.fb)) + C::THREADS - 1) / C::THREADS : 0;
    const int64_t blocks = weight_blocks<C>(j) + scale_blocks + zero_blocks;
    if (blocks > 0x7fffffff) return fail(fn, "too many blocks");
    j.scale_blocks = (unsigned)scale_blocks;
    j.zero_blocks = (unsigned)zero_blocks;
    hipLaunchKernelGGL((vec ? pack_layer_kernel<C, true> : pack_layer_kernel<C, false>), dim3((unsigned)blocks), dim3(C::THREADS), 0, stream, j);
    return launched(fn);
}

// Blocks of 128 columns, but of 64 where there would be few of 128 and where the second on a CU would have it to itself.
// Up to 128 blocks leave CUs without work either way and take as long as a block does: 64 / 128 columns, cold weights, scales and
// zero-points with them, 1024 x 1024 at 2 / 3 / 4 / 8 bits 5.9 / 6.3 / 4.7 / 4.0 against 7.9 / 8.1 / 5.3 / 4.4 us.  144 ... 224 blocks take
// 0 - 10 % less by 128 columns at 2 and 3 bits (4096 x 3072 at 2 12.0 against 10.8), within 3 % at 4 and 8.  More than 256 and up to 384, one and a
// half per CU, 0 - 13 % more: 4096 x 5120 at 2 / 3 bits 18.0 / 19.1 against 19.2 / 20.2, 8192 x 1280 at 4 10.3 / 11.6, 4096 x 1152 at 8 6.3 / 6.9; so do
// 256 of them at 4 and 8 bits, whose scales and zero-points are more blocks in front (4096 x 1024 at 8 5.9 / 6.6), at 2 and 3 they take
// 4 - 8 % less.  Beyond, 128 columns take 4 % less in the mean (4096 x 4096 at 4 15.6 / 14.1; 87 points up to 1536 blocks, 0.87 - 1.08 x).
// Columns loaded one by one are packed by 64 beyond 256 blocks at all: 4096 x 5117 at 2 / 3 / 4 bits 27.7 / 28.7 / 25.0 against 34.7 / 37.3 / 28.2,
// 4096 x 8189 at 2 37.1 against 49.0, 4096 x 3069 at 8 17.1 against 20.1 (60 points 0.97 - 1.37 x, twenty of them within 2 %); 144 ... 256
// blocks are level by either, but 256 at 3 bits 23.1 by 128 columns, 28.1 by 64.
template <int NBITS>
int launch_layer(const char* fn, const PackJob& j, hipStream_t stream) {
    const int64_t wide = weight_blocks<PackCfg<NBITS, 512>>(j);
    const bool vec = j.N % 4 == 0 && (uintptr_t)j.weight % 16 == 0;
    const bool narrow = wide <= 128 || (wide >= (NBITS >= 4 ? 256 : 257) && (wide <= 384 || !vec));
    return narrow ? launch_blocks<PackCfg<NBITS, 256>>(fn, j, vec, stream) : launch_blocks<PackCfg<NBITS, 512>>(fn, j, vec, stream);
}

int launch_layer(const char* fn, const PackJob& j, hipStream_t stream) {
    switch (j.nbits) {
        case 8: return launch_layer<8>(fn, j, stream);
        case 4: return launch_layer<4>(fn, j, stream);
        case 3: return launch_layer<3>(fn, j, stream);
        case 2: return launch_layer<2>(fn, j, stream);
        default: return fail(fn, "nbits must be 2, 3, 4 or 8");
    }
}

// ---------------------------------------------------------------------------------------------
// Calibration kernels
// ---------------------------------------------------------------------------------------------
constexpr int kStreamThreads = 256;
constexpr int kStreamUnroll = 4;

// Every thread requests kStreamUnroll 16-byte units, all before it touches any, and folds them into one word.  The
// word is stored only if it equals a fixed constant, which random data practically never does: the loads cannot
// be dropped and the block ends with its last byte -- no cross-lane sum, no barrier, no store.  (A version that
// wrote one checksum word per block through a wave shuffle and LDS measured 6 % slower at 47 MB: the read ceiling
// is what this kernel is for.)
__global__ __launch_bounds__(kStreamThreads) void stream_read_kernel(const u32x4* __restrict__ src, size_t n16,
                                                                     uint32_t* __restrict__ sink) {
    const size_t per_block = (size_t)kStreamThreads * kStreamUnroll;
    size_t base = (size_t)blockIdx.x * per_block + threadIdx.x;
    uint32_t acc = 0;
    u32x4 v[kStreamUnroll];
#pragma unroll
    for (int u = 0; u < kStreamUnroll; u++) {
        const size_t i = base + (size_t)u * kStreamThreads;
        v[u] = __builtin_nontemporal_load(src + (i < n16 ? i : n16 - 1));
    }
#pragma unroll
    for (int u = 0; u < kStreamUnroll; u++) acc ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
    if (acc == 0x9E3779B9u) sink[blockIdx.x & 4095] = acc;
}

__global__ __launch_bounds__(kStreamThreads) void stream_copy_kernel(u32x4* __restrict__ dst, const u32x4* __restrict__ src,
                                                                     size_t n16) {
    const size_t per_block = (size_t)kStreamThreads * kStreamUnroll;
    size_t base = (size_t)blockIdx.x * per_block + threadIdx.x;
    u32x4 v[kStreamUnroll];
#pragma unroll
    for (int u = 0; u < kStreamUnroll; u++) {
        const size_t i = base + (size_t)u * kStreamThreads;
        if (i < n16) v[u] = __builtin_nontemporal_load(src + i);
    }
#pragma unroll
    for (int u = 0; u < kStreamUnroll; u++) {
        const size_t i = base + (size_t)u * kStreamThreads;
        if (i < n16) __builtin_nontemporal_store(v[u], dst + i);
    }
}

// bf16 -> fp16, eight elements per thread: exact wherever fp16 is normal, magnitudes above 65504 saturate
// (the conversion rounds toward zero), infinities and NaN pass through -- the conversion the quantized-linear
// kernels apply to bf16 activations they read themselves.
__device__ __forceinline__ uint32_t bf16_pair_to_f16_pair(uint32_t v) {
    const float lo = __builtin_bit_cast(float, v << 16);
    const float hi = __builtin_bit_cast(float, v & 0xFFFF0000u);
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo, hi));
}

__global__ __launch_bounds__(256) void bf16_to_f16_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                          int64_t n) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i + 8 <= n) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(src + i);
        *reinterpret_cast<u32x4*>(dst + i) = u32x4{bf16_pair_to_f16_pair(v.x), bf16_pair_to_f16_pair(v.y),
                                                   bf16_pair_to_f16_pair(v.z), bf16_pair_to_f16_pair(v.w)};
    } else {
        for (int64_t j = i; j < n; j++) dst[j] = (uint16_t)bf16_pair_to_f16_pair(src[j]);
    }
}

}  // namespace

extern "C" int qf_version(void) { return 102; }

extern "C" int qf_bf16_to_f16(const uint16_t* src, uint16_t* dst, int64_t n, void* stream_) {
    if (!src || !dst) return fail("qf_bf16_to_f16", "null pointer");
    if (n <= 0) return fail("qf_bf16_to_f16", "n must be positive");
    if (((uintptr_t)src | (uintptr_t)dst) % 16 != 0) return fail("qf_bf16_to_f16", "src and dst must be 16-byte aligned");
    hipLaunchKernelGGL(bf16_to_f16_kernel, dim3((unsigned)((n + 2047) / 2048)), dim3(256), 0, (hipStream_t)stream_, src, dst, n);
    return launched("qf_bf16_to_f16");
}

extern "C" int qf_pack_layer(const int32_t* weight, int8_t* w_out, const uint16_t* scale, uint16_t* s_out, const int32_t* zero,
                             int8_t* z_out, int64_t K, int64_t N, int64_t G, int nbits, uint32_t* bad, void* stream_) {
    const char* fn = "qf_pack_layer";
    if (!weight || !w_out || (scale && !s_out) || (zero && !z_out)) return fail(fn, "null pointer");
    if (K <= 0 || N <= 0 || K % 32 != 0) return fail(fn, "K must be a positive multiple of 32, N positive");
    const int fb = nbits == 3 ? 4 : nbits;
    if ((scale || zero) && G <= 0) return fail(fn, "G must be positive");
    if (nbits != 2 && nbits != 3 && nbits != 4 && nbits != 8) return fail(fn, "nbits must be 2, 3, 4 or 8");
    if (zero && G % (8 / fb) != 0) return fail(fn, "G must fill whole bytes of zero-points");
    return launch_layer(fn, PackJob{weight, (uint32_t*)w_out, scale, s_out, zero, (uint8_t*)z_out, K, N, G, nbits, fb, bad, 0, 0},
                        (hipStream_t)stream_);
}

extern "C" int qf_pack_weight(const int32_t* weight, int8_t* out, int64_t K, int64_t N, int nbits, void* stream_) {
    const char* fn = "qf_pack_weight";
    if (!weight || !out) return fail(fn, "null pointer");
    if (K <= 0 || N <= 0 || K % 32 != 0) return fail(fn, "K must be a positive multiple of 32, N positive");
    return launch_layer(fn, PackJob{weight, (uint32_t*)out, nullptr, nullptr, nullptr, nullptr, K, N, 0, nbits, 8, nullptr, 0, 0},
                        (hipStream_t)stream_);
}

extern "C" int qf_pack_zero(const int32_t* zero, int8_t* out, int64_t G, int64_t N, int nbits, void* stream_) {
    const char* fn = "qf_pack_zero";
    if (!zero || !out) return fail(fn, "null pointer");
    if (nbits != 2 && nbits != 3 && nbits != 4 && nbits != 8) return fail(fn, "nbits must be 2, 3, 4 or 8");
    const int fb = nbits == 3 ? 4 : nbits;
    if (G <= 0 || N <= 0 || G % (8 / fb) != 0) return fail(fn, "G must fill whole bytes of zero-points");
    return launch_layer(fn, PackJob{nullptr, nullptr, nullptr, nullptr, zero, (uint8_t*)out, 0, N, G, nbits, fb, nullptr, 0, 0},
                        (hipStream_t)stream_);
}

extern "C" int qf_transpose_scale(const uint16_t* scale, uint16_t* out, int64_t G, int64_t N, void* stream_) {
    const char* fn = "qf_transpose_scale";
    if (!scale || !out) return fail(fn, "null pointer");
    if (G <= 0 || N <= 0) return fail(fn, "G and N must be positive");
    return launch_layer(fn, PackJob{nullptr, nullptr, scale, out, nullptr, nullptr, 0, N, G, 8, 8, nullptr, 0, 0}, (hipStream_t)stream_);
}

__global__ void empty_kernel(uint32_t* sink) {
    if (sink == nullptr && threadIdx.x == 0xFFFFu) sink[0] = 1;     // never true: the kernel does nothing
}

extern "C" int qf_empty_launch(int64_t blocks, int64_t threads, void* stream_) {
    if (blocks <= 0 || blocks > 0x7fffffff || threads <= 0 || threads > 1024) return fail("qf_empty_launch", "blocks positive, threads in 1..1024");
    hipLaunchKernelGGL(empty_kernel, dim3((unsigned)blocks), dim3((unsigned)threads), 0, (hipStream_t)stream_, (uint32_t*)nullptr);
    return launched("qf_empty_launch");
}

extern "C" int qf_stream_read(const void* src, size_t bytes, uint32_t* sink, void* stream_) {
    if (!src || !sink) return fail("qf_stream_read", "null pointer");
    if (bytes == 0 || bytes % 16 != 0) return fail("qf_stream_read", "bytes must be a positive multiple of 16");
    const size_t n16 = bytes / 16, per_block = (size_t)kStreamThreads * kStreamUnroll;
    hipLaunchKernelGGL(stream_read_kernel, dim3((unsigned)((n16 + per_block - 1) / per_block)), dim3(kStreamThreads), 0,
                       (hipStream_t)stream_, (const u32x4*)src, n16, sink);
    return launched("qf_stream_read");
}

extern "C" int qf_stream_copy(void* dst, const void* src, size_t bytes, void* stream_) {
    if (!dst || !src) return fail("qf_stream_copy", "null pointer");
    if (bytes == 0 || bytes % 16 != 0) return fail("qf_stream_copy", "bytes must be a positive multiple of 16");
    const size_t n16 = bytes / 16, per_block = (size_t)kStreamThreads * kStreamUnroll;
    hipLaunchKernelGGL(stream_copy_kernel, dim3((unsigned)((n16 + per_block - 1) / per_block)), dim3(kStreamThreads), 0,
                       (hipStream_t)stream_, (u32x4*)dst, (const u32x4*)src, n16);
    return launched("qf_stream_copy");
}
