// Dequant-fused low-bit GEMM on the gfx950 matrix cores, one software-pipelined wave per SIMD (from 17 rows on).
//
//   C[m][n] = fp16( sum_k A[m][k] * DQ[n][k] ),   DQ[n][k] = fp16_rn((q[n][k] - Z[n][k/GS]) * s[n][k/GS])
//
// Operands, fragment order and roundings are those of qf_gemm.hip.h (the reference has no matrix-core path,
// qfactory/include/gptq_gemv.h:14-154, and no row count above its register-array size, gptq_gemv.h:34).
//
//   * What bounds it: the MFMAs of a wave and the vector instructions of its dequantisation share the SIMD's issue, and a
//     launch that fills the machine runs at the power limit (1.6 - 1.9 GHz).  So a wave takes as large a tile as it can:
//     MT x 32 activation rows by NT x 32 weight rows, up to 256 x 64 -- 256 accumulators in the accumulation registers and
//     everything else in vector registers -- where a fragment read from LDS serves NT MFMAs and a dequantised weight
//     fragment MT of them.  8192 rows on 12288 x 4096, 4 bits: 749 us with 256 x 32 tiles on two waves per SIMD
//     (qf_gemm.hip.h), 613 us here = 1.35 PFLOP/s; 1024 rows on 22016 x 4096 200 -> 166 us.
//   * Everything reaches LDS by asynchronous buffer loads: activation tiles (BM rows x KI x 128 bytes, PA buffers) and
//     packed weight windows (BN rows x 128 bytes = 1024/NBITS elements, WS buffers), both in the same XOR-swizzled form.
//     No packed word waits in a register on its way, which is what leaves room for the accumulators.
//   * A K-iteration of KI x 64 elements is 4 * KI segments, one MFMA k-step each.  Segment g issues the MFMAs of k-step g,
//     dequantises the weight fragments of g + 1 and reads the activation fragments of g + AHEAD, dealt out behind the
//     MFMAs: nothing is waited for in front of an MFMA.  The one block barrier of an iteration stands in front of the first
//     segment that reads the next tile, not at its end, so the MFMAs of the last AHEAD segments run behind it on registers.
//   * Reuse and arrival: the barrier of iteration t is passed when every wave has read all of tile t (its LDS reads have
//     returned) and its own requests for tile t + 1 have landed.  Between the barriers of t - 1 and t tile t + 2 is
//     requested, into the buffer of tile t - 1, an equal share in every segment (all in the segments of iteration t in
//     front of its barrier, the four waves of a CU asked for more at a time than its address unit takes, and waited to
//     issue: 1 - 4 % of a launch); packed windows in front of the barrier, a window ahead.  The wait allows the requests since
//     the barrier before it to stay in flight and counts nothing else, so loads that the compiler places itself (scales,
//     zero-points) can only make it stricter.
//   * WK groups of waves deal the windows of K between them where a launch has few tiles; their sums meet in LDS.
#pragma once

#include "qf_gemm.hip.h"

namespace qf {

template <int NBITS_, int GS_, bool SYM_, int N_, int K_, int WM_, int WN_, int MT_, int NT_, int KI_, int WK_>
struct GemmWideCfg {
    static constexpr int NBITS = NBITS_, GS = GS_, N = N_, K = K_;
    static constexpr bool SYM = SYM_;
    static constexpr int WM = WM_, WN = WN_;                   // waves along the activation rows and the weight rows
    static constexpr int MT = MT_, NT = NT_;                   // 32-row tiles of a wave in either direction
    static constexpr int WK = WK_;                             // groups of WM x WN waves, each with every WK-th window of K
    static constexpr int WAVES = WM * WN, T = 64 * WAVES * WK; // waves of a group, threads of a block
    static constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN, TN = 32 * NT;
    static constexpr int KI = KI_;                             // 64-element steps of K per iteration (one barrier each)
    static constexpr int SEGS = 4 * KI;                        // segments (MFMA k-steps) of an iteration
    static constexpr int AHEAD = 2;                            // segments between a fragment's read and its MFMAs
    static constexpr int SETS = 4;                             // fragment register sets (SEGS is a multiple)
    static constexpr int SUPK = 1024 / NBITS;                  // elements of K in a 128-byte window
    static constexpr int STEPS = SUPK / 64;                    // 64-element steps of a window
    static constexpr int SUP = STEPS / KI;                     // iterations of a window
    static constexpr int NSUP = K / SUPK;
    static constexpr int NWIN = (NSUP + WK - 1) / WK;          // windows of a group
    static constexpr int ODD = NSUP % WK;                      // != 0: groups ODD .. WK-1 have one window less
    static constexpr int ITERS = NWIN * SUP;
    static constexpr int WS = SUP > 1 ? 2 : 3;                 // window buffers; window P + WS - 1 is requested while P is used
    static constexpr int PA = 3;                               // activation tile buffers
    static constexpr int NGS = SUPK / GS > 0 ? SUPK / GS : 1;  // groups per row and window
    static constexpr int SREGS = (NGS + 1) / 2;
    static constexpr int ZBITS = NGS * NBITS;
    static constexpr int RB = K * NBITS / 8;
    static constexpr int G = K / GS;
    static constexpr int ZRB = G * NBITS / 8;
    static constexpr int GRID_X = (N + BN - 1) / BN;
    static constexpr int A_TILE = KI * BM * 128, W_TILE = BN * 128;           // bytes of one buffer
    static constexpr int AB = KI * BM / 8, WB = BN / 8;        // 1 KB blocks (8 rows) of a buffer: one request of a wave each
    static constexpr int UA = (AB + WAVES - 1) / WAVES;        // requests per wave and tile
    static constexpr int UW = (WB + WAVES - 1) / WAVES;        // ... and window
    static constexpr int PARTS = SUP > 1 ? SUP - 1 : 1;        // a window is requested over that many iterations
    // the epilogue turns a wave's results in LDS: 32*MT rows of its output columns, 16 bytes of padding
    static constexpr int NOUT = QF_GEMM_GATE_UP_SILU ? N / 2 : N;             // output columns of the layer
    static constexpr int TNO = QF_GEMM_GATE_UP_SILU ? TN / 2 : TN;            // ... and of a wave
    static constexpr int OPITCH = TNO * 2 + 16;
    static constexpr size_t LDS_TILES = (size_t)PA * A_TILE + (size_t)WS * W_TILE;
    static constexpr size_t LDS_OUT = (size_t)WAVES * 32 * MT * OPITCH;
    static constexpr size_t LDS_SUMS = (size_t)(WK - 1) * BM * BN * 4;         // the other groups' sums
    static constexpr size_t LDS_END = LDS_SUMS + LDS_OUT;
    static constexpr size_t LDS_BYTES = WK * LDS_TILES > LDS_END ? WK * LDS_TILES : LDS_END;
};

// first of n pieces of work that falls to slot i of `slots`, dealt out evenly from the first slot on
constexpr int wide_first(int i, int n, int slots) { return i < slots ? (i * n + slots - 1) / slots : n; }
// pieces that fall to `part` of `parts` where piece p belongs to part p % parts
constexpr int wide_part(int n, int part, int parts) { return (n - part + parts - 1) / parts; }
// requests for packed words a wave issues in iteration q of a window
template <class C>
constexpr int wide_window_requests(int q) { return q < C::PARTS ? wide_part(C::UW, q, C::PARTS) : 0; }

// 16 bytes per lane from global memory straight into LDS, address = base + per-lane offset + wave-uniform offset: the
// buffer form adds them in the address unit (the flat form costs a 64-bit vector add and a register pair per request)
typedef __amdgpu_buffer_rsrc_t buffer_rsrc;
__device__ __forceinline__ buffer_rsrc rows_from(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0xFFFFFFFF, 0x00020000);
}
__device__ __forceinline__ void buffer_to_lds_16(buffer_rsrc rows, uint32_t lane_offset, uint32_t offset, void* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (__attribute__((address_space(3))) void*)lds, 16, lane_offset, offset, 0, 0);
}

template <class C>
__global__ __launch_bounds__(C::T) void gemm_wide_kernel(
    const uint16_t* __restrict__ A, const uint8_t* __restrict__ W, uint16_t* __restrict__ Cout,
    const uint16_t* __restrict__ S, const uint8_t* __restrict__ Zp, int m_total) {
    constexpr int MT = C::MT, NT = C::NT, SUP = C::SUP, NGS = C::NGS, WAVES = C::WAVES;
    constexpr uint32_t ZMASK = (1u << C::NBITS) - 1u;
    constexpr bool SILU = QF_GEMM_GATE_UP_SILU != 0;

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave_id % WAVES, grp = wave_id / WAVES;
    const int wn = wave % C::WN, wm = wave / C::WN;
    const int li = lane & 31, kb = lane >> 5;
    uint8_t* const tiles = smem + (size_t)grp * C::LDS_TILES;   // the group's buffers
    uint8_t* as_b = tiles;                                      // [PA][KI][BM][128]
    uint8_t* ws_b = tiles + C::PA * C::A_TILE;                  // [WS][BN][128]

    // Block -> tile map: as in qf_gemm.hip.h, the slabs of one column of tiles on one XCD where the generator asks for it
    const int linear = blockIdx.x + gridDim.x * blockIdx.y;
    int col = blockIdx.x, slab = blockIdx.y;
    if (QF_GEMM_XCD_MAP && C::GRID_X >= 8) {
        const int per_group = 8 * gridDim.y;
        const int full = C::GRID_X / 8 * per_group;
        if (linear < full) {
            const int grp8 = linear / per_group, rem = linear % per_group;
            col = grp8 * 8 + rem % 8;
            slab = rem / 8;
        } else {
            constexpr int LAST = C::GRID_X % 8 ? C::GRID_X % 8 : 8;
            const int rem = linear - full;
            col = C::GRID_X / 8 * 8 + rem % LAST;
            slab = rem / LAST;
        }
    }
    const int n_blk = col * C::BN, m_blk = slab * C::BM;
    const int n_wave = n_blk + wn * C::TN;

    // Packed row of the block's local weight row r.  Plain: n_blk + r, clamped to the last row.  Gate+up: local rows
    // 2i, 2i+1 are gate row n_blk/2 + i and its up row N/2 further on, clamped to the last pair.
    auto packed_row = [&](int r) {
        if constexpr (SILU) return min((n_blk + r) >> 1, C::N / 2 - 1) + (r & 1) * (C::N / 2);
        else return min(n_blk + r, C::N - 1);
    };

    // ---- requests: block b of a tile is eight rows of eight 16-byte units; slot 8*row + (c ^ (row/2 % 8)) holds unit c
    //      of the row (no bank conflicts for reads of one unit of 16 rows); blocks past the last repeat it, so that every
    //      wave issues the same number of requests ----
    uint32_t a_off[C::UA];
#pragma unroll
    for (int p = 0; p < C::UA; p++) {
        const int blk = min(p * WAVES + wave, C::AB - 1);      // a buffer holds the iteration's 64-element steps one behind the other
        const int row = (blk % (C::BM / 8)) * 8 + lane / 8, c = (lane % 8) ^ ((row >> 1) & 7);
        a_off[p] = ((uint32_t)min(row, m_total - 1 - m_blk) * C::K + (blk / (C::BM / 8)) * 64 + c * 8) * 2u;   // rows past the end re-read the last one
    }
    const buffer_rsrc a_slab = rows_from(A + (size_t)m_blk * C::K);
    // the group's window w and its iteration `it` in the whole row; past the end the last ones
    auto window_of = [&](int w) { return min(w * C::WK + grp, C::NSUP - 1); };
    // byte offset in a row of the group's iteration `it`: the same for all lanes, and said so: where the compiler had formed it
    // with vector instructions (short rows of K), every request became a loop over the values of the lanes
    auto tile_at = [&](int it) {
        return __builtin_amdgcn_readfirstlane(((uint32_t)window_of(it / SUP) * SUP + (uint32_t)(it % SUP)) * (128u * C::KI));
    };
    auto request_a = [&](int buf, uint32_t at, int p) __attribute__((always_inline)) {
        buffer_to_lds_16(a_slab, a_off[p], at, as_b + (size_t)buf * C::A_TILE + min(p * WAVES + wave, C::AB - 1) * 1024);
    };
    // byte offset of the lane's unit from the block's first packed row (gate+up: from the first gate row; below 4 GiB, checked by the host)
    const int n_first = SILU ? min(n_blk >> 1, C::N / 2 - 1) : min(n_blk, C::N - 1);
    uint32_t w_off[C::UW];
#pragma unroll
    for (int p = 0; p < C::UW; p++) {
        const int row = min(p * WAVES + wave, C::WB - 1) * 8 + lane / 8, c = (lane % 8) ^ ((row >> 1) & 7);
        w_off[p] = (uint32_t)(packed_row(row) - n_first) * C::RB + c * 16;
    }
    const buffer_rsrc w_rows = rows_from(W + (size_t)n_first * C::RB);
    auto window_at = [&](int sup) { return __builtin_amdgcn_readfirstlane((uint32_t)sup * 128u); };      // a scalar operand, as tile_at
    auto request_w = [&](int slot, uint32_t at, int p) __attribute__((always_inline)) {
        buffer_to_lds_16(w_rows, w_off[p], at, ws_b + slot * C::W_TILE + min(p * WAVES + wave, C::WB - 1) * 1024);
    };

    // the first windows and tiles go out before anything else is computed
#pragma unroll
    for (int w = 0; w < C::WS - 1; w++)
        if (w < C::NWIN)
#pragma unroll
            for (int p = 0; p < C::UW; p++) request_w(w, window_at(window_of(w)), p);
#pragma unroll
    for (int p = 0; p < C::UA; p++) request_a(0, tile_at(0), p);
    __builtin_amdgcn_sched_barrier(0);

    // ---- scales and zero-points of the wave's rows, one window in registers and the next on its way ----
    struct Quant { uint32_t s[NT][C::SREGS]; uint32_t z[NT]; };
    uint32_t s_off[NT], z_off[NT];                             // byte offsets from the block's first row
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const uint32_t row = packed_row(wn * C::TN + j * 32 + li) - n_first;
        s_off[j] = row * C::G * 2u;
        z_off[j] = row * C::ZRB;
    }
    const uint8_t* s_rows = reinterpret_cast<const uint8_t*>(S + (size_t)n_first * C::G);
    const uint8_t* z_rows = Zp + (size_t)n_first * C::ZRB;
    auto load_quant = [&](Quant& qu, int sup) {
        const int g0 = sup * C::SUPK / C::GS;
        const uint8_t* sb = s_rows + (size_t)g0 * 2;
        const uint8_t* zb = z_rows + (g0 * C::NBITS) / 8;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const uint8_t* sp = sb + s_off[j];
            if constexpr (NGS == 1) {
                qu.s[j][0] = *reinterpret_cast<const uint16_t*>(sp);
            } else if constexpr (NGS == 2) {
                qu.s[j][0] = *reinterpret_cast<const uint32_t*>(sp);
            } else if constexpr (NGS == 4) {
                const u32x2 v = *reinterpret_cast<const u32x2*>(sp);
                qu.s[j][0] = v.x; qu.s[j][1] = v.y;
            } else {
                const u32x4 v = *reinterpret_cast<const u32x4*>(sp);
                qu.s[j][0] = v.x; qu.s[j][1] = v.y; qu.s[j][2] = v.z; qu.s[j][3] = v.w;
            }
            qu.z[j] = 0;
            if constexpr (!C::SYM) {
                const uint8_t* zp = zb + z_off[j];
                if constexpr (C::ZBITS >= 32) qu.z[j] = *reinterpret_cast<const uint32_t*>(zp);
                else if constexpr (C::ZBITS == 16) qu.z[j] = *reinterpret_cast<const uint16_t*>(zp);
                else if constexpr (C::ZBITS == 8) qu.z[j] = *zp;
                else qu.z[j] = (uint32_t)*zp >> ((g0 * C::NBITS) % 8);
            }
        }
    };
    QConst qc[NT];
    auto make_consts = [&](const Quant& qu, int q, int j) __attribute__((always_inline)) {
        uint32_t sbits, zero;
        if constexpr (C::GS >= C::SUPK) {
            sbits = qu.s[j][0] & 0xFFFFu;
            zero = qu.z[j] & ZMASK;
        } else if constexpr (C::GS >= 64) {
            const int gi = q * 64 / C::GS;
            sbits = (qu.s[j][gi / 2] >> (16 * (gi % 2))) & 0xFFFFu;
            zero = (qu.z[j] >> (gi * C::NBITS)) & ZMASK;
        } else {                                               // GS == 32: group 2q + kb
            sbits = kb ? (qu.s[j][q] >> 16) : (qu.s[j][q] & 0xFFFFu);
            zero = (qu.z[j] >> ((2 * q + kb) * C::NBITS)) & ZMASK;
        }
        if constexpr (C::SYM) zero = 1u << (C::NBITS - 1);
        qc[j] = make_qconst<C::NBITS>((uint16_t)sbits, zero);
    };

    f32x16 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[j][i][v] = 0.0f;

    // fragment addresses: activation row li of a 32-row tile, unit 4*kb + ks; packed row li, the unit that holds the lane's
    // 32 fields of iteration q (8 bits: two units; 2 bits: half a unit)
    const uint32_t sw = (li >> 1) & 7;
    // (units are picked with an XOR of constants into the lane's address; the address is opaque to the compiler where it is
    // used, or every combination is kept in a register of its own through the loop)
    const uint32_t a_lane = (uint32_t)(grp * C::LDS_TILES) + (uint32_t)(wm * MT * 32 + li) * 128 + ((4 * kb) ^ sw) * 16;
    const uint32_t w_lane = (uint32_t)(grp * C::LDS_TILES) + (uint32_t)C::PA * C::A_TILE + (uint32_t)(wn * C::TN + li) * 128
                          + (C::NBITS == 8 ? ((2 * kb) ^ sw) * 16 : C::NBITS == 4 ? (kb ^ sw) * 16 : sw * 16 + 8 * kb);
    auto opaque = [](uint32_t v) __attribute__((always_inline)) {
        asm volatile("" : "+v"(v));
        return v;
    };

    // packed fields of the lane for iteration q of a window: 32 fields = 4*NBITS bytes per tile
    struct Packed { uint32_t w[NT][C::NBITS]; };
    auto read_packed = [&](Packed& pk, uint32_t lane_at, int slot, int q, int j) __attribute__((always_inline)) {
        const uint8_t* tile = smem + slot * C::W_TILE + j * 4096;
        if constexpr (C::NBITS == 2) {
            const u32x2 v = *reinterpret_cast<const u32x2*>(tile + (lane_at ^ (16 * q)));
            pk.w[j][0] = v.x; pk.w[j][1] = v.y;
        } else {
#pragma unroll
            for (int h = 0; h < C::NBITS / 4; h++) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(tile + (lane_at ^ (8 * C::NBITS * q + 16 * h)));
                pk.w[j][4 * h] = v.x; pk.w[j][4 * h + 1] = v.y; pk.w[j][4 * h + 2] = v.z; pk.w[j][4 * h + 3] = v.w;
            }
        }
    };
    f16x8 af[C::SETS][MT], wf[2][NT];
    Packed pk[2];
    auto frags_at = [&](int buf, int seg) __attribute__((always_inline)) {
        return (opaque(a_lane) ^ (16 * (seg % 4))) + (uint32_t)buf * C::A_TILE + (seg / 4) * C::BM * 128;
    };
    auto read_frag = [&](f16x8 (&f)[MT], uint32_t lane_at, int i) __attribute__((always_inline)) {
        f[i] = *reinterpret_cast<const f16x8*>(smem + lane_at + i * 4096);
    };
    // half a weight fragment: four of the lane's eight elements of k-step ks, six or seven instructions
    auto dequant_half = [&](f16x8& f, const Packed& pk, int ks, int j, auto h_tag) __attribute__((always_inline)) {
        constexpr int h = decltype(h_tag)::value;
        const uint32_t word = C::NBITS == 8 ? pk.w[j][2 * ks + h]
                            : C::NBITS == 4 ? pk.w[j][ks]
                            : ks % 2 != 0   ? pk.w[j][ks / 2] >> 8 : pk.w[j][ks / 2];
        const f16x2 v0 = DequantPair<C::NBITS>::template run<2 * h>(word, qc[j]), v1 = DequantPair<C::NBITS>::template run<2 * h + 1>(word, qc[j]);
        f[4 * h] = v0.x; f[4 * h + 1] = v0.y; f[4 * h + 2] = v1.x; f[4 * h + 3] = v1.y;
    };

    // How a segment's work is dealt out behind its MFMAs.  One weight tile per wave: by hand, each MFMA followed by its share
    // and a fence.  More: the scheduler deals out the mix named here -- behind every MFMA a share of the LDS reads and of
    // the vector instructions, the requests at equal distances.  Both ways measured on all tilings, three layers, 32 ... 2048
    // rows: with one weight tile by hand 1 - 7 % less, mean 4 % (half a fragment's six or seven instructions fit behind
    // one MFMA, and the scheduler's groups let them pile up behind the last one); with two and three 2 - 5 % more (there
    // halves leave every second or third MFMA without work and its neighbour with too much).
    auto interleave = [&](auto reads_tag, auto requests_tag) __attribute__((always_inline)) {
        constexpr int MF = MT * NT, VALU = NT * 13 + 4, READS = decltype(reads_tag)::value, REQUESTS = decltype(requests_tag)::value;
        static_for<0, MF>([&](auto i_tag) __attribute__((always_inline)) {
            constexpr int i = decltype(i_tag)::value, here = (i + 1) * REQUESTS / MF - i * REQUESTS / MF;
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                         // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, (READS + MF - 1) / MF, 0);     // LDS reads
            __builtin_amdgcn_sched_group_barrier(0x002, (VALU + MF - 1) / MF, 0);      // vector instructions
            if constexpr (here > 0) __builtin_amdgcn_sched_group_barrier(0x020, here, 0);
        });
        __builtin_amdgcn_sched_barrier(0);
    };

    constexpr bool BY_HAND = NT == 1;
    constexpr int AHEAD = C::AHEAD, SEGS = C::SEGS, KI = C::KI, WS = C::WS, STEPS = C::STEPS;
    constexpr int LAST_BEFORE = SEGS - AHEAD - 1;              // the barrier follows this segment: the next ones read the next tile
    Quant quant[WS];
    auto part_of = [](int g) constexpr { return (g - LAST_BEFORE - 1 + SEGS) % SEGS; };       // segments since the last barrier
    // iteration `it` of the group; s = it % PASS a constant, live 0: nothing to multiply (a group with one window less), left:
    // iterations behind this one, where that is known to be few (tiles and windows past the end are not requested, and the
    // last iteration reads nothing ahead and meets nobody); b0, b1, b2 the buffers of tiles it (and, behind its barrier,
    // it + 3), it + 1 and it + 2
    auto iteration = [&](int it, auto s_tag, auto live_tag, auto left_tag, int b0, int b1, int b2) __attribute__((always_inline)) {
        constexpr int s = decltype(s_tag)::value, left = decltype(left_tag)::value;
        constexpr int q = s % SUP, win = s / SUP;              // iteration of the window; window counted inside a pass
        constexpr bool next_tile = left >= 1, request_tile = left >= 2, request_later = left >= 3, request_window = (left + q) / SUP >= WS - 1;
        constexpr int requests = (request_tile ? C::UA : 0) + (request_window ? wide_window_requests<C>(q) : 0);
        const int sup = it / SUP;
        static_for<0, SEGS>([&](auto g_tag) __attribute__((always_inline)) {
            constexpr int g = decltype(g_tag)::value, step = s * KI + g / 4;
            // what the segment does beside its MFMAs: reads of the fragments of segment g + AHEAD; of the packed words of the next
            // 64-element step, in front of the first segment that dequantises them; the weight fragments of segment g + 1; requests
            constexpr int next = step + 1, next_win = next / STEPS % WS;
            constexpr bool frags_here = next_tile || g + AHEAD < SEGS;
            constexpr bool packed_here = g % 4 == 4 - AHEAD && (next_tile || g + 4 < SEGS);
            constexpr bool dequant_here = g < SEGS - 1 || next_tile, new_step = g % 4 == 3;
            constexpr bool consts_here = dequant_here && new_step && (next % STEPS * 64 % C::GS == 0 || next % STEPS == 0);
            constexpr int reads = (frags_here ? MT : 0) + (packed_here ? NT : 0);
            constexpr int chunks = dequant_here ? (consts_here ? 3 : 2) * NT : 0;
            constexpr int of_tile = (g <= LAST_BEFORE ? request_tile : request_later) ? wide_part(C::UA, part_of(g), SEGS) : 0;
            constexpr int of_window = request_window && g == LAST_BEFORE ? wide_window_requests<C>(q) : 0;
            constexpr int MF = MT * NT;
            uint32_t frags_from = 0, packed_from = 0, tile_from = 0, window_from = 0;
            if constexpr (frags_here) frags_from = g + AHEAD < SEGS ? frags_at(b0, g + AHEAD) : frags_at(b1, g + AHEAD - SEGS);
            if constexpr (packed_here) packed_from = opaque(w_lane);
            if constexpr (of_tile > 0) tile_from = tile_at(g <= LAST_BEFORE ? it + 2 : it + 3);
            if constexpr (of_window > 0) window_from = window_at(window_of(sup + WS - 1));
            if constexpr (request_window && g == 0 && q == 0) load_quant(quant[(win + WS - 1) % WS], window_of(sup + WS - 1));
            static_for<0, MF>([&](auto slot_tag) __attribute__((always_inline)) {
                constexpr int slot = decltype(slot_tag)::value, i = slot / NT, j = slot % NT;
                if constexpr (decltype(live_tag)::value != 0)
                    acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[g % 2][j], af[g % C::SETS][i], acc[j][i], 0, 0, 0);
                static_for<wide_first(slot, reads, MF), wide_first(slot + 1, reads, MF)>([&](auto r_tag) __attribute__((always_inline)) {
                    constexpr int r = decltype(r_tag)::value;
                    if constexpr (packed_here && r < NT) read_packed(pk[next % 2], packed_from, next_win, next % STEPS, r);
                    else read_frag(af[(g + AHEAD) % C::SETS], frags_from, r - (packed_here ? NT : 0));
                });
                static_for<wide_first(slot, chunks, MF), wide_first(slot + 1, chunks, MF)>([&](auto c_tag) __attribute__((always_inline)) {
                    constexpr int per = consts_here ? 3 : 2, tile = decltype(c_tag)::value / per, part = decltype(c_tag)::value % per - (consts_here ? 1 : 0);
                    if constexpr (part < 0) make_consts(quant[next_win], next % STEPS, tile);
                    else dequant_half(wf[(g + 1) % 2][tile], pk[new_step ? next % 2 : step % 2], new_step ? 0 : g % 4 + 1, tile, IntTag<part>{});
                });
                static_for<wide_first(slot, of_tile + of_window, MF), wide_first(slot + 1, of_tile + of_window, MF)>([&](auto r_tag) __attribute__((always_inline)) {
                    constexpr int r = decltype(r_tag)::value;
                    if constexpr (r < of_tile) request_a(g <= LAST_BEFORE ? b2 : b0, tile_from, part_of(g) + r * SEGS);
                    else request_w((win + WS - 1) % WS, window_from, q + (r - of_tile) * C::PARTS);
                });
                if constexpr (BY_HAND) __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (!BY_HAND) interleave(IntTag<(frags_here ? MT : 0) + (packed_here ? NT * (C::NBITS == 8 ? 2 : 1) : 0)>{}, IntTag<of_tile + of_window>{});
            if constexpr (g == LAST_BEFORE && next_tile) {
                wait_loads_and_barrier<QF_GEMM_FULL_DRAIN ? 0 : requests>();
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };

#pragma unroll
    for (int w = 0; w < WS - 1; w++) load_quant(quant[w], window_of(w));
    // tile 1 is younger than all that the first iteration needs and stays in flight over the wait
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (C::ITERS > 1) {
#pragma unroll
        for (int p = 0; p < C::UA; p++) request_a(1, tile_at(1), p);
    }
    wait_loads_and_barrier<QF_GEMM_FULL_DRAIN || C::ITERS < 2 ? 0 : C::UA>();
    static_for<0, NT>([&](auto j_tag) __attribute__((always_inline)) {
        constexpr int j = decltype(j_tag)::value;
        read_packed(pk[0], opaque(w_lane), 0, 0, j);
        make_consts(quant[0], 0, j);
    });
#pragma unroll
    for (int g = 0; g < AHEAD; g++)
#pragma unroll
        for (int i = 0; i < MT; i++) read_frag(af[g], frags_at(0, g), i);
    static_for<0, 2 * NT>([&](auto c_tag) __attribute__((always_inline)) {
        dequant_half(wf[0][decltype(c_tag)::value / 2], pk[0], 0, decltype(c_tag)::value / 2, IntTag<decltype(c_tag)::value % 2>{});
    });
    if constexpr (C::ITERS > 2)
        static_for<LAST_BEFORE + 1, SEGS>([&](auto g_tag) __attribute__((always_inline)) {
#pragma unroll
            for (int p = part_of(decltype(g_tag)::value); p < C::UA; p += SEGS) request_a(2, tile_at(2), p);
        });

    // The accumulators stay in the accumulation registers from here to the stores: left to itself the compiler moves all of
    // them to vector registers behind the loop and, short of those, spills the loop's addresses.
    auto pin = [&]() __attribute__((always_inline)) {
        if constexpr (MT * NT >= 8) {
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int i = 0; i < MT; i++) asm volatile("" : "+a"(acc[j][i]));
        }
    };
    pin();
    // Whole passes (the period of the buffers and register sets) and a straight-line rest, at least as long as the requests
    // run ahead, which also holds the window that some groups do not have: those meet the same barriers and requests without
    // multiplying.
    constexpr int PASS = (WS == 3 ? 6 : 2) * SUP;
    constexpr int REST_MIN = (WS - 2) * SUP + 1 > 3 ? (WS - 2) * SUP + 1 : 3;
    constexpr int FULL_PASSES = C::ITERS > REST_MIN ? (C::ITERS - REST_MIN) / PASS : 0;
    constexpr int REST = C::ITERS - FULL_PASSES * PASS, SHARED = C::ODD != 0 ? SUP : 0;
    int b0 = 0, b1 = 1, b2 = 2;
    auto step = [&](int it, auto s_tag, auto live_tag, auto left_tag) __attribute__((always_inline)) {
        iteration(it, s_tag, live_tag, left_tag, b0, b1, b2);
        const int first = b0;
        b0 = b1; b1 = b2; b2 = first;
    };
    auto rest = [&](auto s_tag, auto live_tag) __attribute__((always_inline)) {
        constexpr int s = decltype(s_tag)::value;
        step(FULL_PASSES * PASS + s, IntTag<s % PASS>{}, live_tag, IntTag<REST - 1 - s>{});
    };
#pragma unroll 1
    for (int pass = 0; pass < FULL_PASSES; pass++)
        static_for<0, PASS>([&](auto s_tag) { step(pass * PASS + decltype(s_tag)::value, s_tag, IntTag<1>{}, IntTag<PASS + REST>{}); });
    static_for<0, REST - SHARED>([&](auto s_tag) { rest(s_tag, IntTag<1>{}); });
    if constexpr (SHARED > 0) {
        if (grp < C::ODD) static_for<REST - SHARED, REST>([&](auto s_tag) { rest(s_tag, IntTag<1>{}); });
        else static_for<REST - SHARED, REST>([&](auto s_tag) { rest(s_tag, IntTag<0>{}); });
    }
    wait_loads_and_barrier<0>();                               // every wave has read its last tile: LDS is free

    pin();

    // ---- the groups' sums meet in LDS (the tiles are no longer needed) ----
    if constexpr (C::WK > 1) {
        constexpr int PER_WAVE = MT * NT * 16 * 64;
        float* sums = reinterpret_cast<float*>(smem + C::LDS_OUT) + (size_t)wave * PER_WAVE + lane * 4;
        if (grp > 0) {
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        *reinterpret_cast<f32x4*>(sums + (size_t)(grp - 1) * WAVES * PER_WAVE + ((j * MT + i) * 4 + v) * 256) =
                            f32x4{acc[j][i][4 * v], acc[j][i][4 * v + 1], acc[j][i][4 * v + 2], acc[j][i][4 * v + 3]};
        }
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int o = 0; o < C::WK - 1; o++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const f32x4 other = *reinterpret_cast<const f32x4*>(sums + (size_t)o * WAVES * PER_WAVE + ((j * MT + i) * 4 + v) * 256);
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[j][i][4 * v + e] += other[e];
                    }
    }

    // ---- store: accumulator register v of a 32x32 tile is (n = 8*(v/4) + 4*(lane/32) + v%4, m = lane%32) ----
    if constexpr (C::NOUT % 4 == 0) {
        // A lane's groups of four go to LDS and come back as 128 (gate+up, one weight tile: 64 or 32) contiguous bytes per
        // row: stored straight from the registers a wave's instruction touches 32 rows with 16 bytes each, and the stores
        // of a 256 x 256 tile took 7 of the 74 us of a round of 64 iterations (8192 rows on 12288 x 4096: 1.14 times the
        // speed of qf_gemm.hip.h on one box with direct stores, 1.17 in this form).
        constexpr int EPU = C::NOUT % 8 == 0 ? 8 : 4;          // elements per store
        constexpr int LPR = C::TNO / EPU, RPI = 64 / LPR;      // lanes per row, rows per instruction
        typedef uint16_t unit_t __attribute__((ext_vector_type(EPU), aligned(8)));
        uint8_t* mine = smem + (size_t)wave * 32 * MT * C::OPITCH;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    uint8_t* at = mine + (i * 32 + li) * C::OPITCH;
                    const float v[4] = {acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]};
                    const int n = j * 32 + 8 * g + 4 * kb;
                    if constexpr (SILU) {
                        // columns n, n+1 and n+2, n+3 are (gate, up) of outputs n/2 and n/2 + 1
                        *reinterpret_cast<uint32_t*>(at + n) = silu_mul_f16(v[0], v[1]) | ((uint32_t)silu_mul_f16(v[2], v[3]) << 16);
                    } else {
                        *reinterpret_cast<u32x2*>(at + 2 * n) = u32x2{f32_to_out_bits(v[0]) | ((uint32_t)f32_to_out_bits(v[1]) << 16),
                                                                      f32_to_out_bits(v[2]) | ((uint32_t)f32_to_out_bits(v[3]) << 16)};
                    }
                }
        __builtin_amdgcn_wave_barrier();
        const int row0 = lane / LPR, c = (lane % LPR) * EPU;
        const int n = (SILU ? n_wave / 2 : n_wave) + c;
        const int m0 = m_blk + wm * MT * 32 + row0;
        uint16_t* dst = Cout + (size_t)m0 * C::NOUT + n;
#pragma unroll 4
        for (int r = 0; r < 32 * MT; r += RPI) {
            // three weight tiles: 12 (or 24, 6) lanes per row leave lanes of the wave, and rows of the last instruction, over
            const bool mine_to_store = (64 % LPR == 0 || row0 < RPI) && ((32 * MT) % RPI == 0 || r + row0 < 32 * MT);
            unit_t v = *reinterpret_cast<const unit_t*>(mine + (mine_to_store ? r + row0 : 0) * C::OPITCH + 2 * c);
            if (mine_to_store && m0 + r < m_total && n < C::NOUT) {
                unit_t* to = reinterpret_cast<unit_t*>(dst + (size_t)r * C::NOUT);
                if constexpr (QF_OUT_ACCUMULATE != 0) {
                    // out = fp16(out + fp16(projection))
                    typedef _Float16 half_t __attribute__((ext_vector_type(EPU)));
                    v = __builtin_bit_cast(unit_t, __builtin_bit_cast(half_t, *to) + __builtin_bit_cast(half_t, v));
                }
                *to = v;
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const int m = m_blk + (wm * MT + i) * 32 + li;
            if (m >= m_total) continue;
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int n = n_wave + j * 32 + 8 * (v / 4) + 4 * kb + v % 4;
                    if (n < C::N) store_out(Cout + (size_t)m * C::N + n, acc[j][i][v]);
                }
        }
    }
}

// Raises the kernel's limit of LDS, once per object (re-entrant: the call is idempotent, the flag only saves repeats).
template <class C>
int gemm_wide_reserve() {
    static std::atomic<bool> reserved{false};
    if (C::LDS_BYTES <= 64 * 1024 || reserved.load(std::memory_order_acquire)) return 0;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_wide_kernel<C>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS_BYTES);
    if (e != hipSuccess) {
        fprintf(stderr, "qfactory gemm: cannot reserve %zu bytes of LDS: %s\n", (size_t)C::LDS_BYTES, hipGetErrorString(e));
        return 2;
    }
    reserved.store(true, std::memory_order_release);
    return 0;
}

template <class C>
int gemm_wide_launch(const void* A, const void* W, void* Cout, const void* S, const void* Zp, int m, hipStream_t stream) {
    const char* why = nullptr;
    if (C::NBITS != 2 && C::NBITS != 4 && C::NBITS != 8) why = "NBITS must be 2, 4 or 8";
    else if (C::WM < 1 || C::WN < 1 || C::MT < 1 || C::NT < 1 || C::WK < 1 || C::T > 1024) why = "block too large";
    else if (C::WK > C::NSUP) why = "a group would own no window";
    else if (C::K % C::SUPK != 0) why = "K must be a whole number of 128-byte windows";
    else if (C::KI < 1 || C::STEPS % C::KI != 0) why = "a window must be whole iterations";
    else if (C::GS <= 0 || C::K % C::GS != 0) why = "GS must divide K";
    else if (C::GS % 32 != 0) why = "a lane's 32 fields must lie inside one group (GS multiple of 32)";
    else if (C::GS < C::SUPK ? C::SUPK % C::GS != 0 : C::GS % C::SUPK != 0) why = "GS must divide 1024/NBITS or be a multiple of it";
    else if (C::NGS > 8 || C::ZBITS > 32) why = "too many groups per 128 packed bytes";
    else if (!C::SYM && (C::G % (8 / C::NBITS)) != 0) why = "K/GS must fill whole zero-point bytes";
    else if (C::LDS_BYTES > 160 * 1024) why = "tiles exceed the 160 KB of LDS";
    else if (C::MT * C::NT * (C::T > 512 ? 4 : C::T > 256 ? 2 : 1) > 16) why = "accumulator tile exceeds the register file";
    else if (QF_GEMM_GATE_UP_SILU && C::N % 8 != 0) why = "gate+up: whole groups of four pairs";
    else if (QF_GEMM_GATE_UP_SILU && QF_OUT_BF16) why = "the SwiGLU epilogue is fp16 only";
    else if (QF_OUT_ACCUMULATE && (QF_OUT_BF16 || QF_GEMM_GATE_UP_SILU)) why = "adding to the output is fp16 only and not combined with the SwiGLU epilogue";
    else if (((size_t)C::N / (QF_GEMM_GATE_UP_SILU ? 2 : 1) + C::BN) * C::RB >= ((size_t)1 << 32) && QF_GEMM_GATE_UP_SILU) why = "gate+up: half the packed weight does not fit a 32-bit row offset";
    if (why) {
        fprintf(stderr, "qfactory gemm: invalid configuration: %s (NBITS=%d GS=%d N=%d K=%d WM=%d WN=%d MT=%d NT=%d KI=%d WK=%d)\n",
                why, C::NBITS, C::GS, C::N, C::K, C::WM, C::WN, C::MT, C::NT, C::KI, C::WK);
        return 1;
    }
    if (m <= 0) return 0;
    if (int rc = gemm_wide_reserve<C>()) return rc;
    dim3 grid(C::GRID_X, (m + C::BM - 1) / C::BM);
    hipLaunchKernelGGL(gemm_wide_kernel<C>, grid, dim3(C::T), C::LDS_BYTES, stream, (const uint16_t*)A, (const uint8_t*)W,
                       (uint16_t*)Cout, (const uint16_t*)S, (const uint8_t*)Zp, m);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        fprintf(stderr, "qfactory gemm: launch failed: %s\n", hipGetErrorString(err));
        return 2;
    }
    return 0;
}

// Two tilings of one problem: Low for launches of at most low_rows rows, C for the others.  The first launch, whatever its
// rows, raises the LDS limit of both kernels: a later one may come under graph capture.
template <class Low, class C>
int gemm_wide_launch_by_rows(const void* A, const void* W, void* Cout, const void* S, const void* Zp, int m, int low_rows,
                             hipStream_t stream) {
    if (m <= 0) return 0;
    if (int rc = gemm_wide_reserve<Low>()) return rc;
    if (int rc = gemm_wide_reserve<C>()) return rc;
    return m <= low_rows ? gemm_wide_launch<Low>(A, W, Cout, S, Zp, m, stream) : gemm_wide_launch<C>(A, W, Cout, S, Zp, m, stream);
}

}  // namespace qf
