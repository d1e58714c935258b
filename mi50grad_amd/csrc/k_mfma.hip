// Multi-query attention over the paged cache with FP16 MFMA (gfx950):
// chunked causal prefill and tree verify.
//
// Semantics: softmax(q K^T / 16) V per query token and head, kv head =
// h*Hkv/H, where new token i of a sequence (slot s_i = len_before + i) sees
//   causal (prefill): keys [0, s_i]  — the reference's rule with the chunk
//       starting after an existing cache (flash_attn_256.hip:78,
//       flash_attn_256_v3.hip:252-255 assume a chunk at position 0);
//   tree:  keys [0, len_before) and the new tokens in its tree bit set
//       (flash_attn_tree.hip:72-175 under tree_attention.py:186-208).
//
// Unit = (sequence, tile of Q new tokens, kv head).  The tile's query rows
// are the Q x G (token, query head) pairs of the GQA group packed row after
// row — every head of the group attends to the same K/V — so W waves of
// 16 x NT rows each (Q = 16*W*NT/G) leave at most G-1 rows idle (the tree
// verify's 9 nodes x 6 heads fill 54 of 64 rows).  Two tiles per wave (256
// rows a unit) halve the LDS reads per product: the LDS pipe carries K and V
// once per wave, and with one tile it is as busy as the matrix pipe.  They
// also double a cut unit's partials, so only steps with enough keys per
// workgroup take them (mq_two_tiles).  Work is split stream-K
// over key blocks (64 keys for prefill steps of eight-wave tiles, 32
// otherwise: mq_keys_for): the blocks of all units are laid end to end, head-major
// (kv head, sequence, tile), and each workgroup takes an equal share, the
// shares dealt out XCD by XCD so the tiles of one (sequence, head) run on
// one XCD and their repeated reads of its keys come from that XCD's L2;
// units cut by a share boundary leave partials for mq_combine_kernel.
//
// K/V blocks travel HBM -> LDS by buffer loads that write LDS directly (no
// register staging), through a ring of LDS stages: four of 32 keys (while
// block i is computed, blocks i+1..i+3, 96 KB, are in flight) or two of 64
// keys (block i+1, 64 KB).  Each wave issues the loads of KEYS/WAVES keys of
// every block; a wave waits for its own loads of block i (vmcnt) and one
// workgroup barrier makes all of them visible and frees the stage of block
// i-1 for the next issue.  Rows are stored with an XOR swizzle of
// their 16-byte granules so both read patterns below are conflict-free.
//
// Per block, wave and 16-row tile t (v_mfma_f32_16x16x32_f16, C layout:
// lane l holds rows 4*(l/16)+i, column l%16):
//   S^T[key][row] = K[key][:] . Q[row][:]   (A = K rows read from LDS once
//       for all NT tiles, B = Q^T held in registers for the whole unit);
//   per row: scale, mask, online softmax (max over the 4 lane groups with
//       two permlane swaps; the reference max moves, and acc is rescaled,
//       only when a block's max passes it by more than a slack), P^T in
//       fp16 — already the B operand of
//   O^T[dim][row] += V^T[dim][key] . P^T[key][row]   (A = V^T read with
//       ds_read_b64_tr_b16 from the row-major V tile; 16 dim tiles).
// The k-index permutation of P^T (keys 4g..4g+3 and 16+4g..16+4g+3 in lane
// group g) is matched by the V^T reads, so the sum is over the right pairs.
#include "k_common.h"
#include "kva_internal.h"

namespace kva {
namespace {

constexpr int kRowBytes = kHeadDim * 2;             // 512 B: one key of one head
constexpr int kPairBytes = 2 * kRowBytes + 32;      // two keys, then 32 B of padding
// LDS stages of the ring for blocks of KEYS keys: 4 x 33 KB or 2 x 66 KB.
template <int KEYS> constexpr int ring_stages() { return KEYS == 32 ? 4 : 2; }
template <int KEYS> constexpr int tile_bytes() { return KEYS / 2 * kPairBytes; }  // K or V of a block
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kStripRow = 128 + 16;  // a row of a wave's epilogue strip: 64 dims, padded


__device__ __forceinline__ int mq_wg_start(int w, int n, int W) { return floor_muldiv(w, n, W); }
__device__ __forceinline__ int mq_wg_of(int p, int n, int W) {
    int w = floor_muldiv(p, W, n);
    while (w + 1 < W && mq_wg_start(w + 1, n, W) <= p) ++w;
    return w;
}
// Largest i in [0, n) with pre[i] <= x (pre non-decreasing, pre[0] <= x;
// wave-uniform arguments).  Each round reads 64 evenly spaced entries of the
// remaining interval with one vector load and keeps the stretch between the
// last entry <= x and the next (a ballot: the entries <= x are a prefix of
// the lanes): two rounds up to 4096 entries, where a binary search by
// scalar loads took one dependent round trip per halving.
__device__ __forceinline__ int upper_index(const int32_t *pre, int n, int x, int lane) {
    int lo = 0, hi = n;  // the answer lies in [lo, hi)
    while (hi - lo > 1) {
        const int step = (hi - lo + 63) >> 6;  // entries between probes
        const int i = lo + lane * step;
        const uint64_t ok = __ballot(i < hi && pre[i] <= x);  // lane 0: pre[lo] <= x
        const int k = ok ? 63 - __clzll(ok) : 0;
        lo = __builtin_amdgcn_readfirstlane(lo + k * step);
        hi = __builtin_amdgcn_readfirstlane(min(hi, lo + step));
    }
    return lo;
}

// LDS layout of a K or V tile: keys in pairs (one 1 KB load each) 1056 B
// apart, and in odd keys the 16-byte granules swapped in twos (K) or fours
// (V).  The padding and the swaps spread both read patterns over all banks
// — K reads take 16 consecutive keys at one granule, V^T reads 4
// consecutive keys at two neighbouring granules — while every read of a
// lane stays at a fixed offset from one base, so the addresses are
// immediates (key = key index within the block).
__device__ __forceinline__ int key_off(int key) { return (key >> 1) * kPairBytes + (key & 1) * kRowBytes; }
__device__ __forceinline__ int k_granule(int key, int p) { return p ^ (key & 1); }
__device__ __forceinline__ int v_granule(int key, int p) { return p ^ ((key & 1) << 2); }

// The facts of one unit (all wave-uniform, read by scalar loads).
struct Unit {
    int u, ub, ue;        // unit index and its global block range [ub, ue)
    int b, h, tile;       // sequence (index in the step), kv head, query tile
    int ctx, ns, tok, T;  // keys visible, first new slot, first token, new tokens
    const int32_t *trow;  // block-table row
};

// Units are head-major: unit u is tile r = u % U1 of head u / U1 (U1 =
// upre[n_seqs], one head's units), and sequence b holds tiles
// [upre[b], upre[b+1]).  b is a hint (a sequence at or before the unit's
// within the same head), so a walk in unit order scans each sequence once.
template <int KEYS>
__device__ __forceinline__ Unit load_unit(const MultiQueryArgs &a, int u, int b) {
    Unit x;
    x.u = u;
    x.ub = ld_uniform(a.mq_pre + u) + kMqUnitCost;  // its first block (positions before: the start cost)
    x.ue = ld_uniform(a.mq_pre + u + 1);
    const int U1 = ld_uniform(a.upre + a.n_seqs);
    x.h = u / U1;
    const int r = u - x.h * U1;
    if (r < ld_uniform(a.upre + b)) b = 0;  // the walk entered the next head
    while (ld_uniform(a.upre + b + 1) <= r) ++b;
    x.b = b;
    x.tile = r - ld_uniform(a.upre + b);
    x.ctx = ld_uniform(a.ctx_lens + b);
    x.ns = ld_uniform(a.new_start + b);
    x.tok = ld_uniform(a.tok_off + b);
    x.T = ld_uniform(a.tok_off + b + 1) - x.tok;
    x.trow = a.table + static_cast<size_t>(ld_uniform(a.seq_ids + b)) * a.table_stride;
    return x;
}

// Page of this wave's keys of block g of unit un (see issue_block), by a
// scalar load: the four-stage ring's.  (Read a block ahead there, at the end
// of the previous block, it measured 10 % slower: the scalar load in flight
// makes every LDS wait of the block drain.  The two-stage ring reads it ahead
// by a vector load, page_ahead in mq_kernel.)
template <int WAVES, int KEYS>
__device__ __forceinline__ int block_page(const Unit &un, int g, bool on, int wv) {
    const int key0 = (g - un.ub) * KEYS + KEYS / WAVES * wv;
    return on ? ld_uniform(un.trow + (min(key0, un.ctx - 1) >> 4)) : 0;
}

// Issue this wave's share of block g of unit un into LDS stage `st`: keys
// kPer*wv .. kPer*wv + kPer-1 of the block (kPer = KEYS/WAVES, within one
// page), K and V, one 1 KB load per two keys each (lane l writes granule
// l%32 of key 2i + l/32).  Keys past the sequence read its last key (finite
// data; the mask drops them).  A disabled issue (past the workgroup's share)
// goes through an empty resource: no memory access, but the same loads, so
// every wave's load counter advances alike.
template <int WAVES, int KEYS>
__device__ __forceinline__ void issue_block(uint8_t *st, const MultiQueryArgs &a, const Unit &un, int g, bool on,
                                            int page, int wv, int lane, int row_bytes) {
    constexpr int kPer = KEYS / WAVES;
    static_assert(kPer <= kBlockTokens && kBlockTokens % kPer == 0, "a wave's keys of a block lie in one page");
    const int key0 = (g - un.ub) * KEYS + kPer * wv;  // key of the unit
    const int last = un.ctx - 1;
    const size_t off = (static_cast<size_t>(page) * kBlockTokens * row_bytes + un.h * kRowBytes) / 2;
    const uint32_t n = on ? kBlockTokens * row_bytes : 0u;
    const auto rk = ro_rsrc(a.k_pool + off, n), rv = ro_rsrc(a.v_pool + off, n);
    const int q = lane & 31;
    if (key0 + kPer - 1 <= last) {
        // All of the wave's keys exist (the sequence's last block aside):
        // rows two apart differ by a scalar offset.
        const int row0 = (key0 & 15) + (lane >> 5);
        const int kl = lane >> 5;  // parity of the key (kPer is even)
        const uint32_t vk = row0 * row_bytes + 16 * k_granule(kl, q), vv = row0 * row_bytes + 16 * v_granule(kl, q);
#pragma unroll
        for (int i = 0; i < kPer / 2; ++i) {
            const uint32_t dst = lds_addr(st + (kPer * wv / 2 + i) * kPairBytes);  // this load's two keys
            load_to_lds_at(rk, dst, vk, 2 * i * row_bytes);
            load_to_lds_at(rv, dst + tile_bytes<KEYS>(), vv, 2 * i * row_bytes);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < kPer / 2; ++i) {
        const int kl = kPer * wv + 2 * i + (lane >> 5);  // key within the block
        const int row = min(key0 + 2 * i + (lane >> 5), last) & 15;
        const uint32_t dst = lds_addr(st + (kPer * wv / 2 + i) * kPairBytes);
        load_to_lds(rk, dst, row * row_bytes + 16 * k_granule(kl, q));
        load_to_lds(rv, dst + tile_bytes<KEYS>(), row * row_bytes + 16 * v_granule(kl, q));
    }
}

// Block i's loads have landed in LDS when at most the loads of the blocks
// issued after it and before this wait (ring stages - 2 of them, KEYS/WAVES
// loads each per wave) are outstanding.
template <int WAVES, int KEYS>
__device__ __forceinline__ void wait_block() { wait_vm<KEYS / WAVES * (ring_stages<KEYS>() - 2)>(); }

__device__ __forceinline__ half8_t as_h8(uint4 v) { return __builtin_bit_cast(half8_t, v); }

// A row's reference max moves only when a block's max exceeds it by more
// than this (log2 units): probabilities then stay below 2^8 (fp16 holds
// them to the same relative precision) and the accumulators are rescaled
// only on such jumps, not at every block where some row's max grew.
constexpr float kRescaleSlack = 8.0f;

// Stream-K share of workgroup i.  Workgroup i runs on XCD i % 8, so with
// W a multiple of 8 the shares are dealt out XCD by XCD: XCD x takes shares
// [x*W/8, (x+1)*W/8), consecutive in unit order.  With head-major units the
// tiles of one (sequence, head), which all read that head's keys, then run
// together on one XCD and share its L2.
__device__ __forceinline__ int mq_share_of(int i, int W) {
    return (W & 7) == 0 ? (i & 7) * (W >> 3) + (i >> 3) : i;
}

// Operands read ahead of the products that use them.  Left alone, the
// compiler reads one operand, waits for it and multiplies: an LDS round trip
// (over 100 cycles) for every 16 to 32 cycles of products.  The scheduling
// barriers pin the order; a ring of operands holds the reads in flight.
// Two tiles per wave, 2048 tokens after 16400: 886 us unpinned, 798 with three
// ahead, 808 with two and 813 with four; one tile per wave 1050 -> 959.  Two
// tiles per wave have no register to spare: 36, 40 and 52 spill with two, three
// and four ahead, none of them inside the products (the unit's start and end,
// the page of the next block).
constexpr int kQkAhead = 3, kPvAhead = 3;

template <int NT, int WAVES, bool TREE, int KEYS>
__global__ __launch_bounds__(64 * WAVES) void mq_kernel(MultiQueryArgs a) {
    constexpr int kRing = ring_stages<KEYS>();
    constexpr int kTileBytes = tile_bytes<KEYS>();
    // Keys folded in at a time: a block's, or with two row tiles per wave
    // half of a 64-key block's (the scores of all would not fit the
    // registers beside two tiles' accumulators).
    constexpr int kFold = NT == 1 ? KEYS : 32;
    constexpr int kKT = kFold / 16;  // 16-key tiles of a fold (QK)
    constexpr int kKS = kFold / 32;  // 32-key steps of a fold (PV)
    __shared__ __attribute__((aligned(16))) uint8_t ring[kRing][2 * kTileBytes];
    __shared__ __attribute__((aligned(16))) uint8_t strips[WAVES][16 * kStripRow];  // the epilogue's, per wave
    const int w = mq_share_of(blockIdx.x, a.n_wg);  // this workgroup's share (and partial slots)
    const int W = a.n_wg;
    const int NB = a.total_blocks;
    const int q0 = mq_wg_start(w, NB, W);
    const int q1 = mq_wg_start(w + 1, NB, W);
    if (q0 >= q1) return;  // uniform over the workgroup
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int col = lane & 15;  // this lane's row within each 16-row tile (C/B column)
    const int grp = lane >> 4;  // lane group: keys 4*grp.. of a 16-key tile
    const int hkv = a.num_kv_heads;
    const int nh = a.num_heads;
    const int G = nh / hkv;
    const int Q = a.q_tile;
    const int row_bytes = hkv * kRowBytes;
    const float scale = kLog2e / 16.0f;

    // The token of this lane's query row in each of the wave's NT tiles.
    int iq[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int rho = 16 * (wv * NT + t) + col;
        iq[t] = rho / G;
    }

    // Issue side: the unit and block of the next load, kRing-1 blocks ahead
    // of the compute side, across unit boundaries.
    const int u0 = upper_index(a.mq_pre, a.n_units, q0, lane);
    const int U1 = ld_uniform(a.upre + a.n_seqs);
    Unit iu = load_unit<KEYS>(a, u0, upper_index(a.upre, a.n_seqs, u0 % U1, lane));
    int ig = max(q0, iu.ub);
    if (ig >= q1) return;  // the share holds only a unit's start cost
    int ipage = 0;  // page of the next issue
    auto fetch_page = [&]() { ipage = block_page<WAVES, KEYS>(iu, ig, ig < q1, wv); };
    // With two stages every load has landed when a block begins, so the
    // page of the next issue can come by a vector load behind this block's:
    // no wait of its own (a scalar load ahead of its use would make every
    // LDS wait of the block drain, scalar loads returning out of order).
    constexpr bool kPageAhead = kRing == 2;
    int vpage = 0;
    auto page_ahead = [&]() {
        const int key0 = (ig - iu.ub) * KEYS + KEYS / WAVES * wv;
        const auto tr = ro_rsrc(iu.trow, static_cast<uint32_t>(a.table_stride) * 4u);
        vpage = static_cast<int>(
            __builtin_amdgcn_raw_buffer_load_b32(tr, ig < q1 ? 4 * (min(key0, iu.ctx - 1) >> 4) : 0, 0, 0));
    };
    auto issue = [&](int slot) {
        const bool on = ig < q1;
        issue_block<WAVES, KEYS>(ring[slot], a, iu, ig, on, ipage, wv, lane, row_bytes);
        if (on && ++ig < q1 && ig >= iu.ue) {
            iu = load_unit<KEYS>(a, iu.u + 1, iu.b);
            ig = iu.ub;
        }
    };
    Unit cu = iu;
    int g = ig;
#pragma unroll
    for (int s = 0; s + 1 < kRing; ++s) {
        fetch_page();
        issue(s);
    }
    if constexpr (kPageAhead) page_ahead();

    int n_done = 0;  // blocks computed by this workgroup (ring position)
    while (true) {
        const int seg_end = min(cu.ue, q1);
        const bool whole = g == cu.ub && seg_end == cu.ue;
        // Query rows of this unit.  Four lanes load 64 contiguous bytes of a
        // row (in the operand layout's lane order, a load's 64 lanes touch
        // 16 rows in 16-byte pieces, at a third of the rate), then a lane
        // permutation gives each lane its operand pieces.  Rows past the
        // unit's tokens read a row that exists; they are never written.
        bool qvalid[NT];
        int qslot[NT];
        uint64_t qbits[NT];
        uint4 qb[NT][8];  // B operand Q^T: dims 32*kk + 8*grp .. +8
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int qi = cu.tile * Q + iq[t];
            qvalid[t] = iq[t] < Q && qi < cu.T;
            qslot[t] = cu.ns + qi;
            qbits[t] = (TREE && qvalid[t]) ? a.tok_bits[cu.tok + qi] : 0ull;
            const int rl = 16 * (wv * NT + t) + (lane >> 2);
            const int il = rl / G, ql = cu.tile * Q + il;
            const bool has = il < Q && ql < cu.T;
            const uint16_t *qr = a.q +
                                 (static_cast<size_t>(cu.tok + (has ? ql : 0)) * nh + cu.h * G + (has ? rl - il * G : 0)) *
                                     kHeadDim +
                                 8 * (lane & 3);
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) qb[t][kk] = ld16(qr + 32 * kk);
            const int from = 4 * (4 * col + grp);  // bytes: the lane that holds this lane's pieces
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
                qb[t][kk].x = __builtin_amdgcn_ds_bpermute(from, qb[t][kk].x);
                qb[t][kk].y = __builtin_amdgcn_ds_bpermute(from, qb[t][kk].y);
                qb[t][kk].z = __builtin_amdgcn_ds_bpermute(from, qb[t][kk].z);
                qb[t][kk].w = __builtin_amdgcn_ds_bpermute(from, qb[t][kk].w);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // Take delivery of the query rows here, once per unit: left to the
        // compiler, the wait for them would sit inside the block loop and
        // (not seeing the LDS loads) drain the ring at every block.
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            asm volatile("" : "+v"(qbits[t]));
#pragma unroll
            for (int kk = 0; kk < 8; ++kk)
                asm volatile("" : "+v"(qb[t][kk].x), "+v"(qb[t][kk].y), "+v"(qb[t][kk].z), "+v"(qb[t][kk].w));
        }
        float m[NT], l[NT];
        float4_t acc[NT][16];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            m[t] = -INFINITY;
            l[t] = 0.0f;
#pragma unroll
            for (int dt = 0; dt < 16; ++dt) acc[t][dt] = float4_t{0.f, 0.f, 0.f, 0.f};
        }

        for (; g < seg_end; ++g) {
            wait_block<WAVES, KEYS>();
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (kPageAhead)
                ipage = __builtin_amdgcn_readfirstlane(vpage);
            else
                fetch_page();
            issue((n_done + kRing - 1) % kRing);
            if constexpr (kPageAhead) page_ahead();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
            for (int fold = 0; fold < KEYS / kFold; ++fold) {
                const uint8_t *kt = ring[n_done % kRing] + fold * (kFold / 2) * kPairBytes;
                const uint8_t *kbase = kt + key_off(col) + 16 * k_granule(col, grp);
                const int key0 = (g - cu.ub) * KEYS + fold * kFold;

                // S^T for keys key0 + 16*nt + 4*grp + i, row `col` of each tile.
                float4_t s[NT][kKT];
#pragma unroll
                for (int nt = 0; nt < kKT; ++nt)
#pragma unroll
                    for (int t = 0; t < NT; ++t) s[t][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
                // Operand i: key tile i % kKT (key 16*nt + col), k-step i / kKT
                // (granule 4*kk + grp): kbase + nt*8 pairs + 64*kk.
                auto read_k = [&](int i) -> uint4 {
                    return *reinterpret_cast<const uint4 *>(kbase + 8 * (i % kKT) * kPairBytes + 64 * (i / kKT));
                };
                uint4 ka[kQkAhead];
#pragma unroll
                for (int i = 0; i < kQkAhead; ++i) ka[i] = read_k(i);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 8 * kKT; ++i) {
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        s[t][i % kKT] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(ka[i % kQkAhead]), as_h8(qb[t][i / kKT]),
                                                                              s[t][i % kKT], 0, 0, 0);
                    if (i + kQkAhead < 8 * kKT) ka[i % kQkAhead] = read_k(i + kQkAhead);
                    __builtin_amdgcn_sched_barrier(0);
                }
                half8_t pb[NT][kKS];
                float corr[NT];
                bool rescale = false;
                // A block wholly before the step's first new slot is visible to
                // every row (wave-uniform test); otherwise mask key by key.  Rows
                // past the unit's tokens are never written, so the open case
                // needs no mask at all.
                const bool open = key0 + kFold <= cu.ns;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    // Masked scores become -inf; the max is taken over the raw
                    // scores and scaled once (scale > 0 keeps the order and the
                    // rounding of the largest), and the probabilities below
                    // fold the scale into one fma.
                    if (!open) {  // wave-uniform: blocks of the cache prefix skip this
#pragma unroll
                        for (int nt = 0; nt < kKT; ++nt)
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                bool vis;
                                if constexpr (TREE) {
                                    // The cache before the step, then the new rows
                                    // in the node's bit set (bits only for the
                                    // step's nodes, so keys past the sequence drop
                                    // out).  Bitwise, so no lane branches.
                                    const int rel = key0 + 16 * nt + 4 * grp + i - cu.ns;
                                    const bool bit = ((qbits[t] >> (rel & 63)) & 1ull) != 0;
                                    vis = qvalid[t] & ((rel < 0) | ((rel < 64) & bit));
                                } else {
                                    // key0 + 16nt + 4grp + i <= qslot (qslot < ctx)
                                    vis = qvalid[t] & (16 * nt + i <= qslot[t] - key0 - 4 * grp);
                                }
                                s[t][nt][i] = vis ? s[t][nt][i] : -INFINITY;
                            }
                    }
                    float mx = -INFINITY;
#pragma unroll
                    for (int nt = 0; nt < kKT; ++nt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[t][nt][i]);
                    mx = group4_max(mx) * scale;
                    // Move the reference max only on a jump past the slack (or
                    // from -inf, where acc and l are still zero).
                    const bool jump = mx > m[t] + kRescaleSlack;
                    const float mn = jump ? mx : m[t];
                    const float mu = (mn == -INFINITY) ? 0.0f : mn;  // rows with nothing visible yet
                    corr[t] = __builtin_amdgcn_exp2f(m[t] - mu);
                    rescale = rescale || (jump && m[t] != -INFINITY);
                    uint32_t pk[2 * kKT];
#pragma unroll
                    for (int nt = 0; nt < kKT; ++nt) {
                        pk[2 * nt] = pack_p2(__builtin_amdgcn_exp2f(fmaf(s[t][nt][0], scale, -mu)),
                                             __builtin_amdgcn_exp2f(fmaf(s[t][nt][1], scale, -mu)));
                        pk[2 * nt + 1] = pack_p2(__builtin_amdgcn_exp2f(fmaf(s[t][nt][2], scale, -mu)),
                                                 __builtin_amdgcn_exp2f(fmaf(s[t][nt][3], scale, -mu)));
                    }
                    // l sums the fp16 probabilities PV uses.
                    constexpr uint32_t kOnes = 0x3c003c00u;  // fp16 pair (1, 1)
                    float psum = 0.0f;
#pragma unroll
                    for (int i = 0; i < 2 * kKT; ++i) psum = dot2(pk[i], kOnes, psum);
                    l[t] = l[t] * corr[t] + psum;
                    m[t] = mn;
#pragma unroll
                    for (int ks = 0; ks < kKS; ++ks)
                        pb[t][ks] = __builtin_bit_cast(half8_t, make_uint4(pk[4 * ks], pk[4 * ks + 1], pk[4 * ks + 2],
                                                                          pk[4 * ks + 3]));
                }
                // Rescale only when some row's reference max moved (wave-uniform).
                if (__builtin_amdgcn_ballot_w64(rescale)) {
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int dt = 0; dt < 16; ++dt) acc[t][dt] *= corr[t];
                }
                // V^T operand of dim tile dt: ds_read_b64_tr_b16 gives lane c of
                // a 16-lane group column c of the 4 x 16 block whose row r the
                // group's lanes 4r..4r+3 address, 8 bytes each: here key
                // 4*grp + r (then 16 + 4*grp + r), dims 16*dt + 4*(lane%4) ...
                // Key 16*hh + 4*grp + vr, granule 2*dt + vs/2: for odd keys the
                // swap of fours moves dims 32*dt.. by +-64 B, + when bit 1 of dt
                // is clear, - when set, so two bases cover every dt.
                const int vr = (lane & 15) >> 2;
                const int vs = lane & 3;
                const uint8_t *vb = kt + kTileBytes + key_off(4 * grp + vr) + 16 * (vs >> 1) + 8 * (vs & 1);
                const uint8_t *vbase[2] = {vb + 64 * (vr & 1), vb - 64 * (vr & 1)};
                // Operand i: dim tile i / kKS, keys 32*(i % kKS) .. (16 pairs on).
                auto read_v = [&](int i) -> half8_t {
                    short4_t part[2];
#pragma unroll
                    for (int hh = 0; hh < 2; ++hh) {
                        const uint8_t *src =
                            vbase[(i / kKS >> 1) & 1] + (16 * (i % kKS) + 8 * hh) * kPairBytes + 32 * (i / kKS);
                        part[hh] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t *)src);
                    }
                    const uint2 v0 = __builtin_bit_cast(uint2, part[0]);
                    const uint2 v1 = __builtin_bit_cast(uint2, part[1]);
                    return __builtin_bit_cast(half8_t, make_uint4(v0.x, v0.y, v1.x, v1.y));
                };
                half8_t va[kPvAhead];
#pragma unroll
                for (int i = 0; i < kPvAhead; ++i) va[i] = read_v(i);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 16 * kKS; ++i) {
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        acc[t][i / kKS] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[i % kPvAhead], pb[t][i % kKS],
                                                                                acc[t][i / kKS], 0, 0, 0);
                    if (i + kPvAhead < 16 * kKS) va[i % kPvAhead] = read_v(i + kPvAhead);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            ++n_done;
        }

        // The four lane groups hold disjoint keys of each row.
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float lt = group4_sum(l[t]);
            const int rho = 16 * (wv * NT + t) + col;
            if (whole) {
                // Through the wave's LDS strip, 64 dims at a time, so that
                // eight lanes hold 128 contiguous bytes of a row: the gate is
                // read and the output written in whole lines (from the
                // accumulator layout, in 32-byte pieces of 16 rows, a unit's
                // end took 2.2 to 5 us).
                const float inv = 1.0f / lt;
                const int r8 = lane >> 3, c8 = lane & 7;  // row (and row + 8) and 16-byte piece
                bool has[2];
                size_t orow[2], grow[2];
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
                    const int rl = 16 * (wv * NT + t) + 8 * hh + r8;
                    const int il = rl / G, ql = cu.tile * Q + il;
                    has[hh] = il < Q && ql < cu.T;
                    const size_t tq = static_cast<size_t>(cu.tok + (has[hh] ? ql : 0));
                    const int hq = cu.h * G + (has[hh] ? rl - il * G : 0);
                    orow[hh] = (tq * nh + hq) * kHeadDim + 8 * c8;
                    grow[hh] = tq * a.gate_stride + hq * kHeadDim + 8 * c8;
                }
                constexpr int kGateAhead = NT == 1 ? 4 : 1;  // strips of gate requested together
                uint4 gw[kGateAhead][2];
                uint8_t *strip = strips[wv];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if (a.gate && c % kGateAhead == 0) {
#pragma unroll
                        for (int k = 0; k < kGateAhead; ++k)
#pragma unroll
                            for (int hh = 0; hh < 2; ++hh) gw[k][hh] = ld16g(a.gate + grow[hh] + 64 * (c + k));
                    }
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const float4_t o = acc[t][4 * c + d] * inv;
                        *reinterpret_cast<uint2 *>(strip + kStripRow * col + 32 * d + 8 * grp) =
                            pack_out4(o[0], o[1], o[2], o[3]);
                    }
#pragma unroll
                    for (int hh = 0; hh < 2; ++hh) {
                        uint4 y = *reinterpret_cast<const uint4 *>(strip + kStripRow * (8 * hh + r8) + 16 * c8);
                        if (a.gate) {
                            const uint2 lo = gate4(make_uint2(y.x, y.y), make_uint2(gw[c % kGateAhead][hh].x, gw[c % kGateAhead][hh].y));
                            const uint2 hi = gate4(make_uint2(y.z, y.w), make_uint2(gw[c % kGateAhead][hh].z, gw[c % kGateAhead][hh].w));
                            y = make_uint4(lo.x, lo.y, hi.x, hi.y);
                        }
                        if (has[hh]) st16(a.out + orow[hh] + 64 * c, y);
                    }
                    if (NT > 1) __builtin_amdgcn_sched_barrier(0);
                }
            } else if (qvalid[t]) {
                // Slot 2w: the unit began at or before this share (its first
                // segment); slot 2w+1: the share's last segment.  (Rows past
                // the tile's tokens are not merged: 10 of a nine-node tree's 64.)
                const int slot = 2 * w + (cu.ub <= q0 ? 0 : 1);
                const size_t rowi = static_cast<size_t>(slot) * (16 * WAVES * NT) + rho;
                float *ar = a.ws_acc + rowi * kHeadDim;
#pragma unroll
                for (int dt = 0; dt < 16; ++dt)
                    *reinterpret_cast<float4 *>(ar + 16 * dt + 4 * grp) =
                        make_float4(acc[t][dt][0], acc[t][dt][1], acc[t][dt][2], acc[t][dt][3]);
                if (grp == 0) {
                    a.ws_ml[rowi * 2] = m[t];
                    a.ws_ml[rowi * 2 + 1] = lt;
                }
            }
        }
        if (g >= q1) break;
        cu = load_unit<KEYS>(a, cu.u + 1, cu.b);
        g = cu.ub;
        if (g >= q1) break;  // the share ends inside the next unit's start cost
    }
    // Loads past the share write LDS too: none may land after the
    // workgroup's LDS is handed on.
    __builtin_amdgcn_s_waitcnt(0);
}

// Merge the partials of units cut across workgroups: a wave per row of a cut
// unit, four dims per lane.  The step plan holds a record per cut unit
// (kva_step_begin finds them from the same shares as the launch), so a wave
// waits for two memory round trips: its record, then every piece's (m, l)
// and acc row (eight at a time) and the row's gate, requested before any is
// used and merged online.  Latency bounds it, so the rows are spread as wide
// as they go: one row per wave and 1 KB per load instruction.  Sixteen rows
// per workgroup, 16 dims per thread and four pieces at a time measured 16.8
// us on 4 x 512 gated tokens and 8.5 on 8 trees of nine nodes.
constexpr int kMqCombineRows = 4;  // rows (waves) per workgroup
__global__ __launch_bounds__(64 * kMqCombineRows) void mq_combine_kernel(MultiQueryArgs a) {
    constexpr int kMaxP = 8;  // pieces requested together
    const int32_t *rec = a.mq_cut + static_cast<size_t>(blockIdx.x) * kMqCutWords;
    const int h = ld_uniform(rec);
    const int tq0 = ld_uniform(rec + 1);      // the tile's first new token (step order)
    const int n_valid = ld_uniform(rec + 2);  // its tokens
    const int w0 = ld_uniform(rec + 3);
    const int w1 = ld_uniform(rec + 4);
    const int slot0 = ld_uniform(rec + 5);
    const int slot_rows = 16 * a.n_waves * a.n_t;
    const int G = a.num_heads / a.num_kv_heads;
    const int rho = __builtin_amdgcn_readfirstlane(kMqCombineRows * blockIdx.y + (threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int iq = __builtin_amdgcn_readfirstlane(rho / G);
    const int gq = rho - iq * G;
    if (iq >= n_valid) return;
    const size_t tq = static_cast<size_t>(tq0 + iq);
    const int hq = h * G + gq;
    const uint2 gw = a.gate ? ld8(a.gate + tq * a.gate_stride + hq * kHeadDim + 4 * lane) : make_uint2(0, 0);
    // Running merge: (big, lt, o) over the pieces so far; m in log2 units.
    float big = -INFINITY, lt = 0.0f;
    float4_t o = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int wb = w0; wb <= w1; wb += kMaxP) {
        float2 ml[kMaxP];
        float4_t v[kMaxP];
#pragma unroll
        for (int i = 0; i < kMaxP; ++i) {
            const int ww = wb + i;
            if (ww <= w1) {
                const int slot = ww == w0 ? slot0 : 2 * ww;
                const size_t rowi = static_cast<size_t>(slot) * slot_rows + rho;
                ml[i] = *reinterpret_cast<const float2 *>(a.ws_ml + rowi * 2);
                v[i] = reinterpret_cast<const float4_t *>(a.ws_acc + rowi * kHeadDim)[lane];
            } else {
                ml[i] = make_float2(-INFINITY, 0.0f);
                v[i] = float4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
        float nb = big;
#pragma unroll
        for (int i = 0; i < kMaxP; ++i) nb = fmaxf(nb, ml[i].x);
        const float mu = (nb == -INFINITY) ? 0.0f : nb;  // rows that see no key of these pieces
        const float keep = (big == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(big - mu);
        lt *= keep;
        o *= keep;
#pragma unroll
        for (int i = 0; i < kMaxP; ++i) {
            const float c = (ml[i].x == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(ml[i].x - mu);
            lt += c * ml[i].y;
            o += c * v[i];
        }
        big = nb;
    }
    const float inv = 1.0f / lt;
    uint2 y = pack_out4(o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv);
    if (a.gate) y = gate4(y, gw);
    *reinterpret_cast<uint2 *>(a.out + (tq * a.num_heads + hq) * kHeadDim + 4 * lane) = y;
}

template <int NT, int WAVES>
hipError_t launch_mq(const MultiQueryArgs &a, hipStream_t s) {
    // 64-key blocks only for eight-wave causal tiles (mq_keys_for).
    const bool k64 = a.keys == 64 && WAVES == 8 && !a.tree;
    if (a.keys != 32 && !k64) return hipErrorInvalidValue;
    if (a.ev_before) {
        const hipError_t e = hipEventRecord(a.ev_before, s);
        if (e != hipSuccess) return e;
    }
    if constexpr (NT > 1) {  // long prefill steps only
        hipLaunchKernelGGL((mq_kernel<NT, WAVES, false, 64>), dim3(a.n_wg), dim3(64 * WAVES), 0, s, a);
    } else if (a.tree) {
        hipLaunchKernelGGL((mq_kernel<NT, WAVES, true, 32>), dim3(a.n_wg), dim3(64 * WAVES), 0, s, a);
    } else if (k64) {
        if constexpr (WAVES == 8)
            hipLaunchKernelGGL((mq_kernel<NT, WAVES, false, 64>), dim3(a.n_wg), dim3(64 * WAVES), 0, s, a);
    } else {
        hipLaunchKernelGGL((mq_kernel<NT, WAVES, false, 32>), dim3(a.n_wg), dim3(64 * WAVES), 0, s, a);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (a.ev_after && (e = hipEventRecord(a.ev_after, s)) != hipSuccess) return e;
    if (a.n_cut > 0) hipLaunchKernelGGL(mq_combine_kernel, dim3(a.n_cut, 16 * WAVES * NT / kMqCombineRows),
                           dim3(64 * kMqCombineRows), 0, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_multi_query(const MultiQueryArgs &a, hipStream_t s) {
    if (a.n_units <= 0 || a.total_blocks <= 0) return hipSuccess;
    const int G = a.num_heads / a.num_kv_heads;
    if (G < 1 || G > kMqMaxGroup || a.num_heads % a.num_kv_heads) return hipErrorInvalidValue;
    if (a.q_tile != mq_tile_tokens(G, a.n_waves, a.n_t)) return hipErrorInvalidValue;
    if (a.n_t == 1 && a.n_waves == 4) return launch_mq<1, 4>(a, s);
    if (a.n_t == 1 && a.n_waves == 8) return launch_mq<1, 8>(a, s);
    if (a.n_t == 2 && a.n_waves == 8 && a.keys == 64 && !a.tree) return launch_mq<2, 8>(a, s);
    return hipErrorInvalidValue;
}

}  // namespace kva
