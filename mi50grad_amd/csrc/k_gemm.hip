// The projections as LDS-tiled MFMA GEMMs (gfx950): Q/K/V with its norm +
// RoPE + append epilogue, and the O-projection with its residual, for every
// step the x-resident form of k_project.hip does not take.
//
// The reference projects a prefill chunk with its batched FP16 GEMM once
// seq_len >= 32 (gemm_fp16_prefill.hip:47, launched through
// _launch_gemm_fp16 at engine.py:3061-3068 into [Q | Q_gate] and [K | V]),
// then normalises, rotates and appends per token.  Here
//   Y[t][n] = sum_k X[t][k] W[n][k]   (X: [T][hidden], W: the stacked
//   weight rows [w_a; w_b], both k-contiguous)
// runs as tiles of BM tokens x BN weight rows in one of three epilogues:
// - head (BN = 256: one head of one kind, Q, Q_gate, K or V): the workgroup
//   holds complete head rows and does the epilogue of proj_finish_kernel
//   itself: each value rounded to fp16 (what the reference's GEMM stores),
//   then Q -> RMSNorm + RoPE -> q_out, Q_gate -> gate_out, K -> RMSNorm +
//   RoPE -> its page slot (and K, V as projected -> kv_out), V -> its page
//   slot.  No [T][N] intermediate and no second launch;
// - out: fp16(sum + residual), one rounding;
// - part: fp32 partials of a slice of hidden, for a finish kernel, where
//   whole tiles would leave most of the 256 CUs idle.
// The O-projection of 2048 tokens (6144 -> 5120) ran as 32 launch pairs of
// the 64-token form, each reading all of W_o: 1023 us; as 256 tiles of
// 128 x 320 in one launch: 137.  181 tokens: Q/K/V 133 -> 53 us (56 tiles of
// 256 x 256 before, 224 of 192 x 128 over two splits now), O-projection
// 102 -> 27.  2048 tokens' Q/K/V: 278 (gemm_pair_kernel).
//
// Main loop.  Eight waves in a WM x (8 / WM) grid, v_mfma_f32_16x16x32_f16
// with W rows as A and tokens as B.  K goes in chunks of 64 through S LDS
// stages: buffer loads write LDS directly, one barrier per chunk, halfway
// through it, makes the next chunk visible and frees this one's stage, and
// each half of a chunk's operands is read from LDS while the other half
// multiplies.  A chunk of 64 k is one whole 128-byte line per row, which the
// load path moves markedly faster than half lines (a 32-wide chunk in four
// stages is slower although more of it is in flight).  Rows sit 128 bytes
// apart in LDS with their 16-byte granules XOR-swizzled (g_swizzle), chosen
// by which global granule each lane fetches, so the 16 rows an MFMA operand
// read touches fall in different banks.
//
// What bounds it.  A CU keeps about 34 KB of cache misses in flight, so its
// loads run at 42 GB/s from HBM and 110-120 GB/s from L2 whatever is asked
// for ahead (measured with 32 to 96 KB requested): small tiles are bound by
// that (touch_line below raises it), large ones by the matrix units, which
// alone hold 1.3-1.5 PFLOP/s on random data here.
//
// Tile order.  Tiles are dealt out XCD by XCD (workgroup i runs on XCD
// i % 8): each XCD takes a contiguous run, so a row tile's weights are read
// by one XCD and reused from its L2 by the token tiles beside each other.
#include <algorithm>
#include <iterator>

#include "k_common.h"
#include "k_normrope.h"
#include "kva_internal.h"

namespace kva {
namespace {

constexpr int kGWaves = 8;
constexpr int kGXcdCus = 32;           // CUs that share an XCD's L2
constexpr int kGKc = 64;               // k per LDS stage: one 128-byte line per row
constexpr int kGRowBytes = kGKc * 2;   // one row of one stage
constexpr int kGGran = kGKc / 8;       // 16-byte granules per row
// The head epilogue's fp16 rows, padded against bank conflicts.
constexpr int kGEpiRow = kHeadDim * 2 + 16;  // 528 B

enum GemmEpilogue {
    kEpiHead,  // a tile row is a head: fp16 rounding, norm + RoPE, outputs, cache rows
    kEpiOut,   // out = fp16(sum + residual)
    kEpiPart,  // fp32 partials [split][token][row] for a finish kernel
};

// A tile of BM tokens x BN weight rows over WM x (8 / WM) waves and S stages;
// AHEAD: chunks between a load and the line touches that precede it (0: none).
template <int BM_, int BN_, int WM_, int S_, int AHEAD_>
struct GTile {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = kGWaves / WM_, S = S_, AHEAD = AHEAD_;
    static constexpr int kWaveTok = BM / WM, kWaveRows = BN / WN;
    static constexpr int kTM = kWaveTok / 16, kTN = kWaveRows / 16;  // MFMA tiles per wave
    static constexpr int kStageX = BM * kGRowBytes, kStageW = BN * kGRowBytes;
    static constexpr int kStage = kStageX + kStageW;
    static constexpr int kLoadsX = kStageX / 1024 / kGWaves;  // 1 KB loads per wave per stage
    static constexpr int kLoadsW = kStageW / 1024 / kGWaves;
    static constexpr int kTouches = AHEAD > 0 ? 2 : 0;
    static constexpr int kLoads = kLoadsX + kLoadsW + kTouches;
    static constexpr int kLoadsMax = kLoadsX > kLoadsW ? kLoadsX : kLoadsW;
    static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "whole MFMA tiles per wave");
    static_assert(BM % 64 == 0 && BN % 64 == 0, "whole loads per wave");
    static_assert(S * kStage <= (160 - 4 - 2) * 1024, "the ring, the token facts and the touches fit the LDS");
};

// The granule swizzle of row r.  The 16 rows one MFMA operand read touches
// at one logical granule must land on distinct 16-byte bank groups whether
// the LDS serves 8 lanes per 128-byte cycle or 16 per 256-byte cycle: two
// 128-byte rows share a 256-byte cycle, so the even rows take granules 0..7
// and the odd rows the same set XORed by 4.  The main loop has no bank
// conflicts (the head epilogue's are 0.3 % of a launch of 2048 tokens).
__device__ __forceinline__ int g_swizzle(int r) { return ((r >> 1) ^ ((r & 1) << 2)) & 7; }

// LDS byte offset of row r's 16-byte granule g within a stage's X or W part.
__device__ __forceinline__ uint32_t g_swz(int r, int g) { return r * kGRowBytes + 16 * (g ^ g_swizzle(r)); }

// Issue one chunk's loads of this wave into `stage`: load j of the wave
// covers LDS granule slots 64*(8*j + wv) + lane of the X part, then of the
// W part; slot p holds row p / 8 at stored granule p % 8, i.e. global
// granule (p % 8) ^ swizzle(row) of that row.  voff[j] is this lane's row
// and granule (the same for X and W); k_byte moves along the row.
template <class T>
__device__ __forceinline__ void g_issue(uint32_t stage, __amdgpu_buffer_rsrc_t rx, __amdgpu_buffer_rsrc_t rw,
                                        const uint32_t (&voff)[T::kLoadsMax], uint32_t k_byte, int wv) {
#pragma unroll
    for (int j = 0; j < T::kLoadsX; ++j) load_to_lds_at(rx, stage + 1024 * (kGWaves * j + wv), voff[j], k_byte);
#pragma unroll
    for (int j = 0; j < T::kLoadsW; ++j)
        load_to_lds_at(rw, stage + T::kStageX + 1024 * (kGWaves * j + wv), voff[j], k_byte);
}

__device__ __forceinline__ half8_t g_h8(uint4 v) { return __builtin_bit_cast(half8_t, v); }

// A workgroup's LDS: the ring of stages, the facts of a head tile's tokens
// (RoPE position, sequence, slot, page id) and the words of lines touched.
template <class T, int EPI>
struct GShared {
    uint8_t ring[T::S * T::kStage];
    int32_t meta[EPI == kEpiHead ? 4 : 1][EPI == kEpiHead ? T::BM : 1];
    uint32_t touched[T::AHEAD > 0 ? kGWaves * 64 : 1];
};

// Workgroup i runs on XCD i % 8: deal each XCD a contiguous run of n tiles.
__device__ __forceinline__ int g_deal(int i, int n) {
    const int xcd = i & 7, q8 = n >> 3, r8 = n & 7;
    return xcd * q8 + min(xcd, r8) + (i >> 3);
}

// One tile: token tile mt (first token t0 within the launch) of the n_mt that
// a row tile has, row tile rt, and with kEpiPart slice `split` of `splits`.
template <class T, int EPI>
__device__ __forceinline__ void gemm_tile(const ProjectArgs &a, GShared<T, EPI> &sh, int t0, int mt, int n_mt, int rt,
                                          int split, int splits) {
    constexpr int kTM = T::kTM, kTN = T::kTN;
    uint8_t *const ring = sh.ring;
    auto &meta = sh.meta;
    const int N = a.n_a + a.n_b;
    const int n0 = rt * T::BN;                     // first stacked weight row
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int hidden = a.hidden;
    const uint32_t row_bytes = static_cast<uint32_t>(hidden) * 2;

    // The tile's tokens' facts, for the epilogue (requested first, used last).
    if constexpr (EPI == kEpiHead) {
        if (threadIdx.x < T::BM) {
            const int t = min(t0 + static_cast<int>(threadIdx.x), a.n_tok - 1);
            const int pos = a.tok_pos[t], seq = a.tok_seq[t], slot = a.tok_slot[t];
            meta[0][threadIdx.x] = pos;
            meta[1][threadIdx.x] = seq;
            meta[2][threadIdx.x] = slot;
            meta[3][threadIdx.x] = a.table[static_cast<size_t>(seq) * a.table_stride + (slot >> 4)];
        }
    }

    const uint16_t *wbase = n0 < a.n_a ? a.w_a + static_cast<size_t>(n0) * hidden
                                       : a.w_b + static_cast<size_t>(n0 - a.n_a) * hidden;
    const uint16_t *xbase = a.x + static_cast<size_t>(t0) * hidden;
    // X rows past the launch's tokens and W rows past the last one read as
    // zeros (the resources' ranges).
    const uint32_t x_bytes = static_cast<uint32_t>(max(0, min(T::BM, a.n_tok - t0))) * row_bytes;
    const uint32_t w_bytes = static_cast<uint32_t>(min(T::BN, N - n0)) * row_bytes;
    const auto rx = ro_rsrc(xbase, x_bytes), rw = ro_rsrc(wbase, w_bytes);
    const auto rx0 = ro_rsrc(xbase, 0u), rw0 = ro_rsrc(wbase, 0u);
    const uint32_t lds0 = lds_addr(ring);
    // This split's chunks of 64 k.
    const int nc_all = hidden / kGKc;
    const int cb = EPI == kEpiPart ? __builtin_amdgcn_readfirstlane(split * nc_all / splits) : 0;
    const int nc = EPI == kEpiPart ? __builtin_amdgcn_readfirstlane((split + 1) * nc_all / splits) - cb : nc_all;
    uint32_t voff[T::kLoadsMax];
#pragma unroll
    for (int j = 0; j < T::kLoadsMax; ++j) {
        const int row = 8 * (kGWaves * j + wv) + (lane >> 3);
        voff[j] = row * row_bytes + 16 * ((lane & 7) ^ g_swizzle(row));
    }
    // Lines touched ahead.  A CU holds about 34 KB of cache misses in flight
    // whatever its loads ask for: 42 GB/s at HBM latency, 110-120 GB/s when
    // the lines are in L2.  The tiles of one XCD that run together share
    // their operands (W: the token tiles of a row tile; X: the row tiles
    // beside it), so each touches its part of the rows of chunk c + AHEAD
    // and the loads themselves find all of them in L2.
    const uint32_t touch0 = lds_addr(sh.touched) + 256 * wv;
    uint32_t toff_w = 0x80000000u, toff_x = 0x80000000u;  // out of range: no access
    if constexpr (T::AHEAD > 0) {
        const int share_w = min(n_mt, kGXcdCus), share_x = max(1, kGXcdCus / n_mt);
        const int row_w = (64 * wv + lane) * share_w + mt % share_w;
        const int row_x = (64 * wv + lane) * share_x + rt % share_x;
        if (share_w > 1 && row_w < T::BN) toff_w = row_w * row_bytes;
        if (share_x > 1 && row_x < T::BM) toff_x = row_x * row_bytes;
    }
    // A chunk past the end goes through empty resources: the same loads, no
    // memory access, so every wave's load counter advances alike.
    auto issue = [&](int c) {
        const bool on = c < nc;
        g_issue<T>(lds0 + (c % T::S) * T::kStage, on ? rx : rx0, on ? rw : rw0, voff,
                   static_cast<uint32_t>(on ? cb + c : 0) * kGRowBytes, wv);
        if constexpr (T::AHEAD > 0) {
            const bool more = c + T::AHEAD < nc;
            const uint32_t k_byte = static_cast<uint32_t>(more ? cb + c + T::AHEAD : 0) * kGRowBytes;
            touch_line(more ? rw : rw0, touch0, toff_w, k_byte);
            touch_line(more ? rx : rx0, touch0, toff_x, k_byte);
        }
    };

    const int wm = wv / T::WN, wn = wv % T::WN;  // this wave's kWaveTok tokens and kWaveRows rows
    const int col = lane & 15, grp = lane >> 4;
    // Weight rows are the MFMA's A operand and tokens its B: lane l holds
    // rows 16*n + 4*(l/16) .. +3 of token 16*m + l%16, four consecutive
    // outputs of one token.
    float4_t acc[kTM][kTN];
#pragma unroll
    for (int m = 0; m < kTM; ++m)
#pragma unroll
        for (int n = 0; n < kTN; ++n) acc[m][n] = float4_t{0.f, 0.f, 0.f, 0.f};

    // Operands of k step ks (32 of a chunk's 64) of the chunk in stage `st`.
    auto read_step = [&](uint4 (&xo)[kTM], uint4 (&wo)[kTN], const uint8_t *st, int ks) {
        const int g = 4 * ks + grp;
#pragma unroll
        for (int n = 0; n < kTN; ++n)
            wo[n] = *reinterpret_cast<const uint4 *>(st + T::kStageX + g_swz(T::kWaveRows * wn + 16 * n + col, g));
#pragma unroll
        for (int m = 0; m < kTM; ++m)
            xo[m] = *reinterpret_cast<const uint4 *>(st + g_swz(T::kWaveTok * wm + 16 * m + col, g));
    };
    auto multiply = [&](const uint4 (&xo)[kTM], const uint4 (&wo)[kTN]) {
#pragma unroll
        for (int m = 0; m < kTM; ++m)
#pragma unroll
            for (int n = 0; n < kTN; ++n)
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(g_h8(wo[n]), g_h8(xo[m]), acc[m][n], 0, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < T::S; ++s) issue(s);
    wait_vm<T::kLoads * (T::S - 1) + T::kTouches>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    uint4 x0[kTM], w0[kTN], x1[kTM], w1[kTN];
    read_step(x0, w0, ring, 0);
    for (int c = 0; c < nc; ++c) {
        read_step(x1, w1, ring + (c % T::S) * T::kStage, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(x0, w0);
        __builtin_amdgcn_sched_barrier(0);
        // This wave has read all of chunk c, and chunk c+1 has landed.
        wait_vm_lds<T::kLoads * (T::S - 2) + T::kTouches>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        issue(c + T::S);
        read_step(x0, w0, ring + ((c + 1) % T::S) * T::kStage, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(x1, w1);
        __builtin_amdgcn_sched_barrier(0);
    }
    // Every load (the dummy ones past the end too) has landed before the
    // LDS is handed on.
    __builtin_amdgcn_s_waitcnt(0);

    const int row0 = n0 + T::kWaveRows * wn + 4 * grp;  // this lane's first output of tile n = 0
    if constexpr (EPI == kEpiPart) {
        float *part = a.part + static_cast<size_t>(split) * a.n_tok * N;
#pragma unroll
        for (int m = 0; m < kTM; ++m) {
            const int t = t0 + T::kWaveTok * wm + 16 * m + col;
            if (t >= a.n_tok) continue;
#pragma unroll
            for (int n = 0; n < kTN; ++n)
                if (row0 + 16 * n < N)
                    *reinterpret_cast<float4_t *>(part + static_cast<size_t>(t) * N + row0 + 16 * n) = acc[m][n];
        }
        return;
    } else if constexpr (EPI == kEpiOut) {
        // One rounding after the residual add; a lane reads its residual
        // before it writes the same bytes, so out may be the residual.
#pragma unroll
        for (int m = 0; m < kTM; ++m) {
            const int t = t0 + T::kWaveTok * wm + 16 * m + col;
            if (t >= a.n_tok) continue;
            const size_t at = static_cast<size_t>(t) * N + row0;
            uint2 r[kTN];
#pragma unroll
            for (int n = 0; n < kTN; ++n)
                r[n] = (a.residual && row0 + 16 * n < N) ? ld8(a.residual + at + 16 * n) : make_uint2(0, 0);
#pragma unroll
            for (int n = 0; n < kTN; ++n) {
                float4_t v = acc[m][n];
                if (a.residual) v += float4_t{lo_f(r[n].x), hi_f(r[n].x), lo_f(r[n].y), hi_f(r[n].y)};
                if (row0 + 16 * n < N)
                    *reinterpret_cast<uint2 *>(a.y_out + at + 16 * n) =
                        make_uint2(pack_h2(v[0], v[1]), pack_h2(v[2], v[3]));
            }
        }
        return;
    } else {
        static_assert(T::BN == kHeadDim, "a head tile holds whole heads");
        static_assert(T::kWaveTok * kGEpiRow <= T::S * T::kStage, "a wave row's epilogue tile must fit the ring");
        __syncthreads();
        const int head = rt;
        const int H = a.num_heads, hkv = a.num_kv_heads;
        const int hw = threadIdx.x >> 5;  // half-wave 0 .. 15
        const int l32 = threadIdx.x & 31;
        const bool is_q = head < H, is_gate = !is_q && head < 2 * H;
        const int kv = head - 2 * H;  // K heads 0..hkv-1, then V heads
        const bool rot = is_q || (!is_gate && kv < hkv);
        uint16_t *epi = reinterpret_cast<uint16_t *>(ring);
        // The norm weights are the same for every row of the tile; each
        // half-wave's cos/sin rows are requested before the tile part is
        // written, so the finish loop waits on none of them row by row.
        constexpr int kRowsPerHw = T::kWaveTok / (2 * kGWaves);
        NormRopeIn nin[kRowsPerHw];
        const uint4 wnorm = rot ? ld16((is_q ? a.q_w : a.k_w) + 8 * l32) : make_uint4(0, 0, 0, 0);
        const int cl = a.half_rot > 0 ? min(l32, a.half_rot / 4 - 1) : 0;
        // One wave row's tokens at a time: its waves write their sums as
        // fp16 (each rounded once: what the reference's GEMM stores) into
        // the tile [kWaveTok tokens][256 rows], then every wave finishes the
        // part's token rows.
        for (int part = 0; part < T::WM; ++part) {
#pragma unroll
            for (int j = 0; j < kRowsPerHw; ++j) {
                nin[j].w = wnorm;
                nin[j].c = make_uint2(0, 0);
                nin[j].s = make_uint2(0, 0);
                if (rot && a.half_rot > 0) {
                    // Tokens past the launch's end carry the last token's
                    // position, so these reads stay inside the tables.
                    const size_t off =
                        static_cast<size_t>(meta[0][part * T::kWaveTok + hw + 2 * kGWaves * j]) * a.half_rot;
                    nin[j].c = ld8(a.cos_tab + off + 4 * cl);
                    nin[j].s = ld8(a.sin_tab + off + 4 * cl);
                }
            }
            if (wm == part) {
#pragma unroll
                for (int m = 0; m < kTM; ++m)
#pragma unroll
                    for (int n = 0; n < kTN; ++n)
                        *reinterpret_cast<uint2 *>(epi + (16 * m + col) * (kGEpiRow / 2) + T::kWaveRows * wn + 16 * n +
                                                   4 * grp) =
                            make_uint2(pack_h2(acc[m][n][0], acc[m][n][1]), pack_h2(acc[m][n][2], acc[m][n][3]));
            }
            __syncthreads();
            // Finish: one 32-lane group per token row, 8 dims per lane, the
            // arithmetic of proj_finish_kernel (norm_rope_apply: the same bits).
#pragma unroll
            for (int j = 0; j < kRowsPerHw; ++j) {
                const int rr = hw + 2 * kGWaves * j;
                const int r = part * T::kWaveTok + rr;
                const int t = t0 + r;
                if (t >= a.n_tok) break;
                const uint4 y = *reinterpret_cast<const uint4 *>(epi + rr * (kGEpiRow / 2) + 8 * l32);
                if (is_gate) {
                    if (a.gate_out) st16(a.gate_out + (static_cast<size_t>(t) * H + head - H) * kHeadDim + 8 * l32, y);
                    continue;
                }
                if (!is_q && a.kv_out)
                    st16(a.kv_out + (static_cast<size_t>(t) * 2 * hkv + kv) * kHeadDim + 8 * l32, y);
                const uint4 o = rot ? norm_rope_apply<32>(y, nin[j], a.half_rot, a.eps, l32) : y;
                if (is_q) {
                    st16(a.q_out + (static_cast<size_t>(t) * H + head) * kHeadDim + 8 * l32, o);
                    continue;
                }
                const int slot = meta[2][r], blk = meta[3][r];
                const size_t row_base = (static_cast<size_t>(blk) * kBlockTokens + (slot & 15)) * hkv;
                if (kv < hkv)
                    st16(a.k_pool + (row_base + kv) * kHeadDim + 8 * l32, o);
                else
                    st16(a.v_pool + (row_base + kv - hkv) * kHeadDim + 8 * l32, y);
            }
            __syncthreads();  // the part's rows are read before the next part overwrites them
        }
    }
}

template <class T, int EPI>
__global__ __launch_bounds__(64 * kGWaves) void gemm_kernel(ProjectArgs a) {
    __shared__ __attribute__((aligned(16))) GShared<T, EPI> sh;
    const int n_rt = (a.n_a + a.n_b + T::BN - 1) / T::BN;
    const int n_mt = (a.n_tok + T::BM - 1) / T::BM;
    const int splits = EPI == kEpiPart ? a.splits : 1;
    const int tau = g_deal(blockIdx.x, n_rt * splits * n_mt);
    // Token tiles fastest, then row tiles, then splits, so that the tiles
    // beside each other share a row tile's weights and a split's slice of x.
    // (readfirstlane: quotients are computed in vector registers, and the
    // loads' resources must be scalar.)
    const int ws = __builtin_amdgcn_readfirstlane(tau / n_mt);
    const int mt = tau - ws * n_mt;
    const int split = EPI == kEpiPart ? __builtin_amdgcn_readfirstlane(ws / n_rt) : 0;
    gemm_tile<T, EPI>(a, sh, mt * T::BM, mt, n_mt, ws - split * n_rt, split, splits);
}

// Head tiles of two heights in one launch: tiles of TA's tokens for whole
// rounds of the chip, then tiles of TB's for the rest.  Tiles of one height
// leave the last round part empty: 2048 tokens of 5120 -> 14336 are 448 tiles
// of 256 x 256, 1.75 rounds of 256 CUs, 298 us; 256 of those and 256 of
// 192 x 256 take 278.  1300 tokens 268 -> 224 (192 and 128 against 616 tiles
// of 128), 4000 618 -> 523.  Row tile r has k token
// tiles of TA, k = p.hi for the first p.heads rows and p.lo after
// them, and as many of TB as its other tokens need.
template <class TA, class TB>
__global__ __launch_bounds__(64 * kGWaves) void gemm_pair_kernel(ProjectArgs a, GemmPair p) {
    static_assert(TA::BN == kHeadDim && TB::BN == kHeadDim, "head tiles");
    __shared__ __attribute__((aligned(16))) union {
        GShared<TA, kEpiHead> a;
        GShared<TB, kEpiHead> b;
    } sh;
    const int i = blockIdx.x;
    const bool tall = i < p.tall;
    const int tau = tall ? g_deal(i, p.tall) : g_deal(i - p.tall, p.all - p.tall);
    const int hi = tall ? p.hi : p.rest_hi, lo = tall ? p.lo : p.rest_lo;  // tiles of a row tile
    const bool first = tau < p.heads * hi;
    const int rel = first ? tau : tau - p.heads * hi;
    const int per = max(1, first ? hi : lo);
    const int row = __builtin_amdgcn_readfirstlane(rel / per);
    const int mt = rel - row * per;
    const int rt = first ? row : p.heads + row;
    if (tall)
        gemm_tile<TA, kEpiHead>(a, sh.a, mt * TA::BM, mt, per, rt, 0, 1);
    else
        gemm_tile<TB, kEpiHead>(a, sh.b, (first ? p.hi : p.lo) * TA::BM + mt * TB::BM, mt, per, rt, 0, 1);
}

using Tile256x256 = GTile<256, 256, 2, 2, 0>;
using Tile192x256 = GTile<192, 256, 2, 2, 0>;
using Tile128x256 = GTile<128, 256, 2, 3, 1>;
using Tile64x256 = GTile<64, 256, 1, 3, 1>;
using Tile128x320 = GTile<128, 320, 2, 2, 1>;
using Tile256x128 = GTile<256, 128, 4, 3, 1>;
using Tile192x128 = GTile<192, 128, 4, 3, 1>;
using Tile128x128 = GTile<128, 128, 2, 4, 1>;
using Tile64x128 = GTile<64, 128, 1, 6, 1>;

template <class T, int EPI>
hipError_t launch_gemm(const ProjectArgs &a, hipStream_t s) {
    const int n_rt = (a.n_a + a.n_b + T::BN - 1) / T::BN, n_mt = (a.n_tok + T::BM - 1) / T::BM;
    const int splits = EPI == kEpiPart ? a.splits : 1;
    hipLaunchKernelGGL((gemm_kernel<T, EPI>), dim3(n_rt * splits * n_mt), dim3(64 * kGWaves), 0, s, a);
    return hipGetLastError();
}

template <class TA, class TB>
hipError_t launch_pair(const ProjectArgs &a, const GemmPair &p, hipStream_t s) {
    hipLaunchKernelGGL((gemm_pair_kernel<TA, TB>), dim3(p.all), dim3(64 * kGWaves), 0, s, a, p);
    return hipGetLastError();
}

// The tile shapes, and what a 64-wide k chunk of each takes on a full chip
// (us, measured at hidden 5120 and 6144).
struct GemmForm {
    int bm, bn;
    float chunk_us;
    bool head, out, part;  // epilogues built for it
    hipError_t (*launch_head)(const ProjectArgs &, hipStream_t);
    hipError_t (*launch_out)(const ProjectArgs &, hipStream_t);
    hipError_t (*launch_part)(const ProjectArgs &, hipStream_t);
};
const GemmForm kForms[] = {
    {256, 256, 1.88f, true, false, false, launch_gemm<Tile256x256, kEpiHead>, nullptr, nullptr},
    {192, 256, 1.50f, true, false, false, launch_gemm<Tile192x256, kEpiHead>, nullptr, nullptr},
    {128, 256, 1.05f, true, true, true, launch_gemm<Tile128x256, kEpiHead>, launch_gemm<Tile128x256, kEpiOut>,
     launch_gemm<Tile128x256, kEpiPart>},
    {64, 256, 0.84f, true, false, true, launch_gemm<Tile64x256, kEpiHead>, nullptr, launch_gemm<Tile64x256, kEpiPart>},
    {128, 320, 1.30f, false, true, false, nullptr, launch_gemm<Tile128x320, kEpiOut>, nullptr},
    {256, 128, 0.96f, false, true, true, nullptr, launch_gemm<Tile256x128, kEpiOut>,
     launch_gemm<Tile256x128, kEpiPart>},
    {192, 128, 0.76f, false, true, true, nullptr, launch_gemm<Tile192x128, kEpiOut>,
     launch_gemm<Tile192x128, kEpiPart>},
    {128, 128, 0.64f, false, true, true, nullptr, launch_gemm<Tile128x128, kEpiOut>,
     launch_gemm<Tile128x128, kEpiPart>},
    {64, 128, 0.60f, false, true, true, nullptr, launch_gemm<Tile64x128, kEpiOut>, launch_gemm<Tile64x128, kEpiPart>},
};

// The heights that gemm_pair_kernel is built for: indices into kForms.
struct GemmPairForm {
    int tall, low;
    hipError_t (*launch)(const ProjectArgs &, const GemmPair &, hipStream_t);
};
const GemmPairForm kPairs[] = {
    {0, 1, launch_pair<Tile256x256, Tile192x256>},
    {0, 2, launch_pair<Tile256x256, Tile128x256>},
    {1, 2, launch_pair<Tile192x256, Tile128x256>},
};

// Tall tiles for whole rounds of the chip, shared out over n_rt row
// tiles as evenly as leaves the fewest low ones (room: workgroups of those
// rounds).  The search stays within kPairSpread tiles of an even share: over
// 65 to 12000 tokens and 14, 28 and 56 row tiles no plan is estimated slower
// than with the whole range searched, which takes the host 5 ms at 32768
// tokens and grows with their cube; this takes 6 to 9 us from 4096 on.
constexpr int kPairSpread = 8;
constexpr int kPairRounds = 4;  // counts of tall rounds tried, from the most down
GemmPair pair_tiles(int T, int n_rt, int bm, int bm_low, int64_t room) {
    GemmPair best{0, 0, 0, 0, 0, 0, 0};
    const int most = T / bm;
    const int even = static_cast<int>(std::min<int64_t>(most, room / n_rt));
    for (int lo = std::max(0, even - kPairSpread); lo <= even; ++lo) {
        for (int hi = lo + 1; hi <= std::min(most, lo + kPairSpread); ++hi) {
            const int64_t more = (room - static_cast<int64_t>(n_rt) * lo) / (hi - lo);
            const int heads = static_cast<int>(std::min<int64_t>(n_rt, more));
            const int rest_hi = (T - hi * bm + bm_low - 1) / bm_low, rest_lo = (T - lo * bm + bm_low - 1) / bm_low;
            const int tall = heads * hi + (n_rt - heads) * lo;
            const int all = tall + heads * rest_hi + (n_rt - heads) * rest_lo;
            if (tall > 0 && (best.all == 0 || all - tall < best.all - best.tall))
                best = GemmPair{tall, all, heads, hi, lo, rest_hi, rest_lo};
        }
    }
    return best;
}

}  // namespace

// The tile and the split of hidden for T tokens: the least estimated time.
// A round of tiles (one per CU) costs its chunks plus about 3 us to start
// and end, and no less than the operands take to stream at 5 TB/s shared by
// all CUs (48 tokens of 6144 -> 5120 take 20.6 us over four splits, 160
// workgroups, and 17.7 over six, 240); a split adds its partials, written and read back, and the finish launch.  The
// estimate is within 15 % of the measured times it was fitted to (64 to 2048
// tokens of 5120 -> 14336 and 6144 -> 5120, and their halves and quarters):
// 2048 tokens of 6144 -> 5120 take 124 us in 128 x 320 tiles (one round of
// 256), 162 in 192 x 128 (two rounds); over hidden 1536 to 6144, 3072 to 7168
// rows and 1300 to 4096 tokens the 128 x 320 tile takes 10 to 28 % less than
// the next best wherever it is chosen: its rounds come out full; 181 take 22 us in 192 x 128
// over six splits, 29 in 128 x 128 over three, 69 unsplit, and their Q/K/V 46
// us in 192 x 128 over two splits against 59 in 128 x 256 (a tile that holds
// every token reads each weight row once).  With a.hold only partials do, of
// one slice or several.
bool plan_gemm(const ProjectArgs &a, bool heads, int n_cu, size_t part_floats, ProductPlan &plan) {
    const int T = a.n_tok, N = a.n_a + a.n_b;
    if (a.hidden % kGKc != 0 || T > kBigProjMaxTokens || (heads && N % kHeadDim != 0)) return false;
    const int nc = a.hidden / kGKc;
    const double stream_us = 2.0 * a.hidden * (static_cast<double>(N) + T) / 5.0e6;
    ProductPlan best{};
    best.form = best.pair = -1;
    double best_us = 0;
    for (int i = 0; i < static_cast<int>(std::size(kForms)); ++i) {
        const GemmForm &f = kForms[i];
        // Row offsets within a tile are 32-bit.
        if (static_cast<uint64_t>(std::max(f.bm, f.bn)) * 2u * static_cast<uint32_t>(a.hidden) > 0xffffffffull) continue;
        if (heads && a.n_a % f.bn != 0) continue;  // a tile never straddles the two weights
        const double tiles = static_cast<double>((N + f.bn - 1) / f.bn) * ((T + f.bm - 1) / f.bm);
        for (int splits = 1; splits <= kGemmMaxSplits && splits <= nc; ++splits) {
            const bool partial = splits > 1 || a.hold;
            if (partial ? !f.part : !(heads ? f.head : f.out)) continue;
            const double part = static_cast<double>(splits) * T * N;
            if (partial && part > static_cast<double>(part_floats)) break;
            const double rounds = static_cast<double>((static_cast<int64_t>(tiles * splits) + n_cu - 1) / n_cu);
            const double walk = rounds * ((nc + splits - 1) / splits) * f.chunk_us;
            // A CU streams its share of the operands: fewer workgroups than
            // CUs stretch that time.  A tenth of the lesser term is a
            // tie-break (a smaller tile walks the same stream more lightly).
            const double fill = tiles * splits < n_cu ? n_cu / (tiles * splits) : 1.0;
            const double stream = stream_us * fill;
            double us = 3.0 * rounds + (walk > stream ? walk + 0.1 * stream : stream + 0.1 * walk);
            if (partial) us += 4.0 + 8.0 * part / 5.0e6;
            if (best.form < 0 || us < best_us) {
                best.form = i;
                best.splits = splits;
                best.partial = partial;
                best_us = us;
            }
        }
    }
    if (best.form < 0) return false;
    best.bm = kForms[best.form].bm;
    best.bn = kForms[best.form].bn;
    // Two heights, where one leaves its last round part empty.
    for (int i = 0; i < static_cast<int>(std::size(kPairs)); ++i) {
        const GemmPairForm &f = kPairs[i];
        const GemmForm &ft = kForms[f.tall], &fl = kForms[f.low];
        if (!heads || best.partial || a.n_a % ft.bn != 0) break;
        const int n_rt = N / ft.bn;
        const int64_t round = static_cast<int64_t>(n_cu) * ft.bm;
        const int rounds = static_cast<int>((static_cast<int64_t>(T) * n_rt + round - 1) / round);
        for (int r = std::max(1, rounds - kPairRounds); r < rounds; ++r) {
            const GemmPair cut = pair_tiles(T, n_rt, ft.bm, fl.bm, static_cast<int64_t>(r) * n_cu);
            if (cut.all <= cut.tall) continue;
            const int more = (cut.all - cut.tall + n_cu - 1) / n_cu;
            const double walk = nc * (r * ft.chunk_us + more * fl.chunk_us);
            const double us = 3.0 * (r + more) + (walk > stream_us ? walk + 0.1 * stream_us : stream_us + 0.1 * walk);
            if (us < best_us) {
                best.pair = i;
                best.cut = cut;
                best.bm = ft.bm;
                best.bn = ft.bn;
                best.low = fl.bm;
                best_us = us;
            }
        }
    }
    plan = best;
    return true;
}

hipError_t launch_gemm_project(const ProjectArgs &a, bool heads, const ProductPlan &plan, hipStream_t s) {
    if (plan.pair >= 0) return kPairs[plan.pair].launch(a, plan.cut, s);
    const GemmForm &form = kForms[plan.form];
    if (plan.partial) return form.launch_part(a, s);
    return (heads ? form.launch_head : form.launch_out)(a, s);
}

}  // namespace kva
