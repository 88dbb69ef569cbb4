// libqfactory_hip.so, third translation unit: causal attention of a prompt's positions over the KV cache of a
// Llama-style layer.  The entry point is declared in include/qfactory_hip_ext.h.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <stdint.h>

#include "qfactory_hip_ext.h"

namespace {

typedef _Float16 f16;
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

int fail(const char* fn, const char* why) {
    fprintf(stderr, "%s: %s\n", fn, why);
    return 1;
}

// One wave's 32 queries, key by key: two lanes (kb = 0, 1) per query, each with half of the dims.
template <int HD>
__device__ __forceinline__ void attend_by_key(const f16* q_row, const f16* k_rows, const f16* v_rows, f16* dst, int kb, bool have,
                                              int my_pos, int last, float scale_log2) {
    constexpr int UNITS = HD / 16;                                          // eight dims each
    f16x8 qh[UNITS];
    float o[HD / 2], m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int u = 0; u < UNITS; u++) qh[u] = *reinterpret_cast<const f16x8*>(q_row + kb * (HD / 2) + 8 * u);
#pragma unroll
    for (int d = 0; d < HD / 2; d++) o[d] = 0.0f;
#pragma unroll 1
    for (int key = 0; key <= last; key++) {
        const size_t at = (size_t)key * HD + kb * (HD / 2);
        float score = 0.0f;
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            const f16x8 kh = *reinterpret_cast<const f16x8*>(k_rows + at + 8 * u);
#pragma unroll
            for (int e = 0; e < 8; e++) score += (float)qh[u][e] * (float)kh[e];
        }
        score = (score + __shfl_xor(score, 32, 64)) * scale_log2;
        if (key > my_pos) continue;
        const float m_new = fmaxf(m, score), base = m_new == -INFINITY ? 0.0f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - base), p = __builtin_amdgcn_exp2f(score - base);
        m = m_new;
        l = l * alpha + p;
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            const f16x8 vh = *reinterpret_cast<const f16x8*>(v_rows + at + 8 * u);
#pragma unroll
            for (int e = 0; e < 8; e++) o[8 * u + e] = o[8 * u + e] * alpha + p * (float)vh[e];
        }
    }
    if (!have) return;
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        f16x8 r;
#pragma unroll
        for (int e = 0; e < 8; e++) r[e] = (f16)(o[8 * u + e] / l);
        *reinterpret_cast<f16x8*>(dst + kb * (HD / 2) + 8 * u) = r;
    }
}

// ---------------------------------------------------------------------------------------------
// One block: 128 query rows of one (sequence, head), four waves of 32, over key tiles of 64 positions; on the matrix
// cores (v_mfma_f32_32x32x16_f16), scores, running maximum and sums in fp32.
//
//   * The scores are formed transposed, S^T = K Q^T: a lane ends with sixteen keys of ONE query (column lane % 32; its
//     partner lane ^ 32 has the other sixteen), so the softmax is arithmetic inside a lane and one exchange, and
//     the probabilities already are the B operand of O^T += V^T P^T -- the contraction order of an MFMA is free, the
//     fragments of V^T are read to match: keys 16 s + 4 kb .. + 3 and 16 s + 8 + 4 kb .. + 3.  No probability moves between lanes.
//   * Probabilities enter the second product as fp16(p) + fp16(p - fp16(p)), off by at most max(2^-22 p, 2^-25) (the second
//     half is subnormal below p = 1/4): the product costs twice the MFMAs, which are idle otherwise.
//   * A key that a query must not see has probability 0, but 0 times an infinity or NaN in its V still reaches the sum.  A
//     wave with a sum that is not finite (finite values cannot overflow fp32 here) goes through its keys once more, key by
//     key, and leaves out what a query does not see.  The look at the sums costs 0 - 1.5 % (8 x 128 positions 11.2 -> 11.4 us);
//     a look at every V on its way to LDS cost 9 - 17 %, a second pass of the block that shares the registers 3 - 15 %.
//   * K tiles go to LDS as rows, V tiles turned to [dim][key] in 4 x 4 pieces on the way (registers); the next tile is
//     loaded while this one is used.
//
// Bound by memory and by the few dependent trips to it: 8 sequences x 32 heads x 128 positions of 128 dims are 34 MB of
// q, k, v and output, 6 us at the rate of a large copy; 13.5 us here, 45.6 for the library's masked attention over all 256
// positions of the cache (which this reads only up to the last query's).
// ---------------------------------------------------------------------------------------------
constexpr int kRows = 128, kKeys = 64, kThreads = 256;

template <int HD>
__global__ __launch_bounds__(kThreads) void prefill_attention_kernel(
    const f16* __restrict__ q, const f16* __restrict__ k_cache, const f16* __restrict__ v_cache,
    const int64_t* __restrict__ pos, f16* __restrict__ out, int tokens, int heads, int max_len, float scale_log2) {
    constexpr int KSTEPS = HD / 16, DT = HD / 32;
    constexpr int K_PITCH = HD * 2 + 16, V_PITCH = kKeys * 2 + 8;           // bytes
    constexpr int K_UNITS = kKeys * HD / 8 / kThreads;                      // 16-byte units per thread and tile
    constexpr int V_UNITS = (kKeys / 4) * (HD / 4) / kThreads;              // 4 x 4 pieces per thread and tile
    __shared__ __attribute__((aligned(16))) uint8_t ks[kKeys * K_PITCH];
    __shared__ __attribute__((aligned(16))) uint8_t vs[HD * V_PITCH];
    __shared__ int wave_last[kThreads / 64];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 31, kb = lane >> 5;
    const int h = blockIdx.y, b = blockIdx.z;
    const int row = blockIdx.x * kRows + wave * 32 + li;                    // this lane's query
    const bool have = row < tokens;
    const int my_pos = have ? (int)pos[row] : -1;
    const size_t head = ((size_t)b * heads + h) * max_len;                  // first cache row of the (sequence, head)

    // last key of the wave and of the block
    int last = min(my_pos, max_len - 1);
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1) last = max(last, __shfl_xor(last, o, 64));
    if (lane == 0) wave_last[wave] = last;

    f16x8 qf[KSTEPS];
    const f16* q_row = q + (((size_t)b * tokens + min(row, tokens - 1)) * heads + h) * HD;
#pragma unroll
    for (int s = 0; s < KSTEPS; s++) qf[s] = *reinterpret_cast<const f16x8*>(q_row + 16 * s + 8 * kb);
    __syncthreads();
    int block_last = wave_last[0];
#pragma unroll
    for (int w = 1; w < kThreads / 64; w++) block_last = max(block_last, wave_last[w]);

    u32x4 k_reg[K_UNITS];
    u32x2 v_reg[V_UNITS][4];
    auto load_tile = [&](int key0) {
#pragma unroll
        for (int u = 0; u < K_UNITS; u++) {
            const int unit = u * kThreads + tid, key = min(key0 + unit / (HD / 8), max_len - 1);      // past the cache: masked below
            k_reg[u] = *reinterpret_cast<const u32x4*>(k_cache + (head + key) * HD + (unit % (HD / 8)) * 8);
        }
#pragma unroll
        for (int u = 0; u < V_UNITS; u++) {
            const int unit = u * kThreads + tid, d = (unit % (HD / 4)) * 4, key = key0 + unit / (HD / 4) * 4;
#pragma unroll
            for (int e = 0; e < 4; e++)
                v_reg[u][e] = *reinterpret_cast<const u32x2*>(v_cache + (head + min(key + e, max_len - 1)) * HD + d);
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (int u = 0; u < K_UNITS; u++) {
            const int unit = u * kThreads + tid;
            *reinterpret_cast<u32x4*>(ks + (unit / (HD / 8)) * K_PITCH + (unit % (HD / 8)) * 16) = k_reg[u];
        }
#pragma unroll
        for (int u = 0; u < V_UNITS; u++) {
            const int unit = u * kThreads + tid, d = (unit % (HD / 4)) * 4, key = unit / (HD / 4) * 4;
#pragma unroll
            for (int e = 0; e < 4; e++) {                                   // dim d + e of the four keys
                const uint32_t sel = e % 2 ? 0x07060302u : 0x05040100u;
                const uint32_t a = e < 2 ? v_reg[u][0].x : v_reg[u][0].y, c = e < 2 ? v_reg[u][1].x : v_reg[u][1].y;
                const uint32_t f = e < 2 ? v_reg[u][2].x : v_reg[u][2].y, g = e < 2 ? v_reg[u][3].x : v_reg[u][3].y;
                *reinterpret_cast<u32x2*>(vs + (d + e) * V_PITCH + key * 2) =
                    u32x2{__builtin_amdgcn_perm(c, a, sel), __builtin_amdgcn_perm(g, f, sel)};
            }
        }
    };

    f32x16 o[DT];
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int v = 0; v < 16; v++) o[d][v] = 0.0f;
    float m = -INFINITY, l = 0.0f;                                          // l: this lane's keys only, the partner's are added at the end

    if (block_last >= 0) load_tile(0);
    for (int key0 = 0; key0 <= block_last; key0 += kKeys) {                 // block-uniform
        __syncthreads();
        store_tile();
        __syncthreads();
        if (key0 + kKeys <= block_last) load_tile(key0 + kKeys);
        if (key0 > last) continue;                                          // wave-uniform: nothing visible to this wave
        f32x16 sc[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
            for (int v = 0; v < 16; v++) sc[t][v] = 0.0f;
#pragma unroll
            for (int s = 0; s < KSTEPS; s++) {
                const f16x8 kf = *reinterpret_cast<const f16x8*>(ks + (t * 32 + li) * K_PITCH + 32 * s + 16 * kb);
                sc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[s], sc[t], 0, 0, 0);
            }
        }
        // register v of tile t is key key0 + 32 t + 8 (v / 4) + 4 kb + v % 4 of this lane's query
        float top = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int key = key0 + 32 * t + 8 * (v / 4) + 4 * kb + v % 4;
                sc[t][v] = key <= my_pos && key < max_len ? sc[t][v] * scale_log2 : -INFINITY;
                top = fmaxf(top, sc[t][v]);
            }
        const float m_new = fmaxf(m, fmaxf(top, __shfl_xor(top, 32, 64)));
        const float base = m_new == -INFINITY ? 0.0f : m_new;               // nothing visible yet: every p below is 0
        const float alpha = __builtin_amdgcn_exp2f(m - base);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                sc[t][v] = __builtin_amdgcn_exp2f(sc[t][v] - base);
                l += sc[t][v];
            }
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int v = 0; v < 16; v++) o[d][v] *= alpha;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            f16x8 hi, lo;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float p = sc[s / 2][8 * (s % 2) + e];
                hi[e] = (f16)p;
                lo[e] = (f16)(p - (float)hi[e]);
            }
#pragma unroll
            for (int d = 0; d < DT; d++) {
                const uint8_t* at = vs + (d * 32 + li) * V_PITCH + (16 * s + 4 * kb) * 2;
                const f16x4 v0 = *reinterpret_cast<const f16x4*>(at), v1 = *reinterpret_cast<const f16x4*>(at + 16);
                const f16x8 vf = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
                o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, hi, o[d], 0, 0, 0);
                o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, lo, o[d], 0, 0, 0);
            }
        }
    }
    f16* dst = out + (((size_t)b * tokens + row) * heads + h) * HD;
    float look = 0.0f;                                                      // NaN where a sum is not finite
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int v = 0; v < 16; v++) look = __builtin_fmaf(o[d][v], 0.0f, look);
    if (__builtin_expect(__any(have && look != 0.0f), 0)) {
        attend_by_key<HD>(q_row, k_cache + head * HD, v_cache + head * HD, dst, kb, have, my_pos, last, scale_log2);
        return;
    }
    if (!have) return;
    const float inv = 1.0f / (l + __shfl_xor(l, 32, 64));
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int g = 0; g < 4; g++)
            *reinterpret_cast<f16x4*>(dst + 32 * d + 8 * g + 4 * kb) =
                f16x4{(f16)(o[d][4 * g] * inv), (f16)(o[d][4 * g + 1] * inv), (f16)(o[d][4 * g + 2] * inv), (f16)(o[d][4 * g + 3] * inv)};
}

}  // namespace

extern "C" int qf_prefill_attention(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const int64_t* pos,
                                    uint16_t* out, int64_t batch, int64_t tokens, int64_t heads, int64_t head_dim,
                                    int64_t max_len, void* stream_) {
    const char* fn = "qf_prefill_attention";
    if (!q || !k_cache || !v_cache || !pos || !out) return fail(fn, "null pointer");
    if (batch <= 0 || tokens <= 0 || heads <= 0 || max_len <= 0) return fail(fn, "batch, tokens, heads and max_len must be positive");
    if (head_dim != 64 && head_dim != 128) return fail(fn, "head_dim must be 64 or 128");
    if (batch > 65535 || heads > 65535 || tokens > (1 << 30) || max_len > (1 << 30)) return fail(fn, "too many sequences, heads or positions");
    if (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) % 16 != 0) return fail(fn, "tensors must be 16-byte aligned");
    const dim3 grid((unsigned)((tokens + kRows - 1) / kRows), (unsigned)heads, (unsigned)batch);
    const float scale_log2 = 1.4426950408889634f / sqrtf((float)head_dim);
    hipLaunchKernelGGL((head_dim == 64 ? prefill_attention_kernel<64> : prefill_attention_kernel<128>), grid, dim3(kThreads), 0,
                       (hipStream_t)stream_, (const f16*)q, (const f16*)k_cache, (const f16*)v_cache, pos, (f16*)out, (int)tokens,
                       (int)heads, (int)max_len, scale_log2);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        fprintf(stderr, "%s: launch failed: %s\n", fn, hipGetErrorString(err));
        return 2;
    }
    return 0;
}
