// Flash prefill / chunked prefill attention on gfx950 (causal and sliding window).
//
// Replaces the reference's fav2::flash_v2_kernel (kernels/attention_flash_v2.cuh:104-259) and, for long query
// runs, flash_attn2bs_p1(_custom)_kernel (kernels/attention_flash.cuh:28-217).
//
// Work decomposition. A workgroup holds a tile of rows: tokens x the GRP q-heads of one KV head (token-major), so every
// K/V byte it fetches serves the whole GQA group. A work item is one tile of consecutive tokens, or, for short causal
// prompts, the pair of half tiles (i, n-1-i) over the union of their key ranges, so that the keys of the short half are
// fetched once for both and every workgroup carries about the same work (a T=1024 prompt at 8 KV heads is 256 such
// workgroups). choose_plan picks the tile and the form from the launch's sizes. Work items of one (sequence, KV head)
// are mapped onto as few XCDs as the number of heads allows (workgroups are dispatched round-robin over the 8 XCDs), so
// that head's K/V stays in one L2.
//
// Keys are walked in steps of SK keys at absolute positions; each wave takes the NSUB 16-key sub-tiles of its key
// group in a step (one wave per key group and row group). K and V of a step go from HBM/L2 straight into LDS
// with gfx950 direct-to-LDS buffer loads (no staging registers; the buffer range makes rows past the last key
// read as zeros), two stages, one barrier per step. The LDS rows are unpadded and their 16-byte slots are
// XOR-swizzled by the key (kswz, vswz). Each wave then
//   * computes S^T = K Q^T for its rows on 16x16x32 MFMA (K fragments from LDS, Q fragments in registers),
//   * masks (causal / window; a wave-uniform test picks the unmasked fast path) and runs the online softmax in
//     registers over all its keys of the step (a row lives in 4 lanes; the running max moves lazily, so the
//     accumulator is rescaled on few steps),
//   * computes O^T += V^T P^T on 16x16x32 MFMA over its two sub-tiles at once (16x16x16 at HD 512) with V^T
//     read transposed from LDS (ds_read_b64_tr_b16) and P^T straight from the softmax registers.
// At the end the two key-group states of each row are merged through LDS.
//
// Determinism and chunk invariance: step boundaries are absolute, the key group of a sub-tile depends only on
// its position, a sub-tile a row does not attend leaves the row's state exactly unchanged, and the merge order is
// fixed. A row's bits therefore depend only on its query, position and keys - not on the other rows of its tile,
// the tile pairing or how the prompt is chunked (attention_flash_v2.cuh:13-18).
//
// Key splits (kv_split > 0) restrict each work item to the keys of one absolute split and write LSE partials for
// launch_combine. VER is the form for short query runs over long caches (verify, draft trees): the items are the key
// chunks of a ragged batch, found on the device, and the mask takes the tree's ancestor bits (attention_flash.cuh:177).
#include "attn_device.h"
#include "attn_internal.h"
#include <algorithm>
#include <atomic>
#include <climits>
#include <type_traits>

namespace dgx {

struct PrefArgs {
    Problem p;
    Partials part;
    int kv_split;      // 0: none
    uint32_t split_m;  // div_magic(kv_split)
    int nht;           // half tiles (pair) or tiles per sequence
    int nsplit;        // key splits per sequence
    int tqh;           // tokens per half tile (pair) or per tile
    int pair;          // 1: a work item is the half-tile pair (i, nht-1-i); 0: one tile of all the workgroup's rows
    int nitems;        // work items per (sequence, kv head)
    int heads;         // sequences x KV heads
    int grp;           // q-heads per KV head
    float sl2;         // scale * log2(e)
    int fold;          // 1: fold each XCD's slots (two co-resident workgroups per CU take a long and a short item)
    int q_al;          // Q is 16-byte aligned
    int grp_mul;       // ceil(65536 / GRP): rho / GRP = rho * grp_mul >> 16 for rho < 128
    int slots;         // verify: workgroups per (KV head, tile) that run at once
    int ways;          // XCDs that share one KV head's items (> 0), or minus the KV heads that share an XCD; 0: neither
};

// A workgroup is RG x KG waves. RB: 16-row blocks per wave; RG: row groups (waves splitting the tile's rows, the first
// half of them on a pair's first half tile); KG: key groups (waves splitting each step's keys); NS: LDS stages; NSUB:
// 16-key sub-tiles per wave and step.
template <int HD, int RB, int RG, int KG_, int NSUB_>
struct PrefCfg {
    static constexpr int KG = KG_, NW = RG * KG_, NT = NW * 64, NSUB = NSUB_;
    static constexpr int KT = 16 * NSUB;                 // keys per wave per step (NSUB 16-key sub-tiles)
    static constexpr int SK = KG * KT;                   // keys per step
    static constexpr int RR = RG * RB * 16;              // rows per workgroup tile
    static constexpr int HR = RR / 2;                    // rows per half tile
    static constexpr int KS = HD / 32;                   // QK k-steps (16x16x32)
    static constexpr int DB = HD / 16;                   // PV output dim blocks (16x16x16)
    static constexpr int DO = DB / KG;                   // output dim blocks each key group finishes
    static constexpr int SLOTS = HD / 8;                 // 16-byte slots per key row
    static constexpr int ROWB = HD * 2;                  // bytes per key row (16-bit operands)
    static constexpr int HALF = SK * ROWB;               // bytes of one K (or V) step tile
    static constexpr int STAGE = 2 * HALF;               // K, then V, of one step
    static constexpr int NQL = RR * SLOTS / 64 / NW;     // 16-byte Q loads per thread
    static constexpr int NLR = SK * SLOTS / 64;          // 64-slot rows of a step tile (one per wave load)
    static constexpr int NLD = (NLR + NW - 1) / NW;      // 16-byte loads per thread per step (K and V each)
    static constexpr size_t LDS_TILES = (size_t)2 * STAGE;
    static constexpr int XSTR = HD / KG + 4;             // merge exchange row stride (floats)
    // merge exchange: [row block][row group][owner key group][sender slot (KG-1)][16 rows][XSTR]
    static constexpr size_t LDS_MERGE = (size_t)RB * RG * KG * (KG - 1) * 16 * XSTR * 4;
    static constexpr size_t LDS_STATS = (size_t)2 * NW * RB * 16 * 4;
    // The merge statistics follow the exchange, over the tiles; verify runs put both past stage 0, which the next chunk's
    // first step fills meanwhile.
    static constexpr size_t merge_off(bool ver) { return ver ? STAGE : 0; }
    static constexpr size_t lds(bool ver) {
        return LDS_TILES > merge_off(ver) + LDS_MERGE + LDS_STATS ? LDS_TILES : merge_off(ver) + LDS_MERGE + LDS_STATS;
    }
    static constexpr size_t LDS = lds(false);
    static_assert((SK * SLOTS) % 64 == 0, "step loads");
    static_assert((RR * SLOTS) % (64 * NW) == 0 && RR * ROWB <= STAGE && HR % (64 / SLOTS) == 0, "Q tile in a stage");
    static_assert(NSUB == 2 || (NSUB == 1 && RB == 1), "row block layout");
    static_assert((KG == 2 || KG == 4) && DB % KG == 0, "key groups");
};

// Slot swizzles of key row k: 16-byte column c of key k sits in slot c ^ swz(k). V rows use vswz, a permutation of
// the low 4 key bits (keys 0-7 to the even slots, 8-15 to the odd ones), which spreads the 8 keys x 2 columns that
// the 32 lanes of a half V transpose read (keys 4g..4g+3 for g = 0, 1 or g = 2, 3) over all 16 slots of a 256-byte
// bank row. K rows are read 16 bytes per lane by key (lane = key, column 4 ks + g): kswz(k) = k puts the 8 (16)
// keys of a lane group on distinct bank quads (vswz, with its even slots for keys 0-7, measured 4 conflict cycles
// per read there).
__device__ __forceinline__ int vswz(int k) { return ((k & 7) << 1) | ((k >> 3) & 1); }
__device__ __forceinline__ int kswz(int k) { return k & 15; }

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void glb_void;

// LDS reads at addr + OFF that the caller waits for with lds_wait: 16 bytes per lane, and the transpose read.
template <int OFF> __device__ __forceinline__ void lds_read16(u32x4 &d, unsigned addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(d) : "v"(addr), "n"(OFF) : "memory");
}
template <int OFF> __device__ __forceinline__ void lds_read_tr(u32x2 &d, unsigned addr) {
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(d) : "v"(addr), "n"(OFF) : "memory");
}
// Wait until at most CNT younger LDS reads are in flight; the registers in r are written by older ones.
template <int CNT, class T, int N>
__device__ __forceinline__ void lds_wait(T (&r)[N]) {
    static_assert(N == 2 || N == 4 || N == 8, "read batch");
    if constexpr (N == 2)
        asm volatile("s_waitcnt lgkmcnt(%[c])" : "+v"(r[0]), "+v"(r[1]) : [c] "n"(CNT) : "memory");
    else if constexpr (N == 4)
        asm volatile("s_waitcnt lgkmcnt(%[c])" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]) : [c] "n"(CNT) : "memory");
    else
        asm volatile("s_waitcnt lgkmcnt(%[c])" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]),
                     "+v"(r[6]), "+v"(r[7]) : [c] "n"(CNT) : "memory");
}

// One work item: the rows of tile (or pair) qi from the last of (sequence, KV head) over key split sp. Verify runs (whose
// sequence is at position p0) call it for the splits [c0, c1) in turn: the first call loads the Q fragments qop, each call but the last requests the first step
// of the next split before it merges.
template <int HD, int RB, int RG, int KG_, int NSUB, int KVT, int QT, int OT, bool VER, bool FAR>
__device__ __forceinline__ void prefill_item(const PrefArgs &a, int seq, int p0, int kvh, int qi, int sp, int c0, int c1,
                                             u32x4 (&qop)[RB][HD / 32], unsigned char *smem) {
    using Cf = PrefCfg<HD, RB, RG, KG_, NSUB>;
    constexpr int KG = Cf::KG, SK = Cf::SK, KS = Cf::KS, DB = Cf::DB, NLD = Cf::NLD, DO = Cf::DO;
    constexpr int SLOTS = Cf::SLOTS, ROWB = Cf::ROWB, HR = Cf::HR;
    constexpr bool F16 = OpIsF16<KVT>::value;
    constexpr bool DMA = KVT != DT_FP32;                 // 16-bit caches go straight to LDS
    using KE = typename Elem<KVT>::T;
    using QE = typename Elem<QT>::T;
    unsigned char *const xmem = smem + Cf::merge_off(VER);
    float *stm = reinterpret_cast<float *>(xmem + Cf::LDS_MERGE), *stl = stm + Cf::NW * RB * 16;

    const Problem &p = a.p;
    const int GRP = a.grp;

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, ln = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave / KG, kg = wave % KG;
    const size_t krow = (size_t)p.NKV * HD;
    const KE *Kb = kv_base<KE>(p, false, seq) + (size_t)kvh * HD;
    const KE *Vb = kv_base<KE>(p, true, seq) + (size_t)kvh * HD;
    // Prefill tokens are consecutive: token t of this sequence sits at position pbase + t.
    const int pbase = VER ? p0 : __builtin_amdgcn_readfirstlane(p.pos_arr ? p.pos_arr[seq] : p.base);

    // The work item's tokens: one tile, or two half tiles (longest first; an empty half has tok1 == tok0).
    const bool pair = !VER && a.pair, split = VER || a.kv_split > 0;    // (verify items are single tiles over one chunk)
    const int ht0 = a.nht - 1 - qi, ht1 = pair && qi < ht0 ? qi : -1;
    int tok0[2], tok1[2];
    tok0[0] = ht0 * a.tqh; tok1[0] = min(p.T, tok0[0] + a.tqh);
    tok0[1] = ht1 < 0 ? 0 : ht1 * a.tqh; tok1[1] = ht1 < 0 ? 0 : min(p.T, tok0[1] + a.tqh);
    // Keys of the workgroup: the union of both halves' ranges (the first half holds the latest tokens).
    int j_lo = win_lo(pbase + tok0[0], p.window);
    if (tok1[1] > tok0[1]) j_lo = min(j_lo, win_lo(pbase + tok0[1], p.window));
    const int hi_b = pbase + tok1[0];                                   // one past the last key (clamp bound)
    int j_hi = hi_b;
    if (split) { j_lo = max(j_lo, sp * a.kv_split); j_hi = min(j_hi, (sp + 1) * a.kv_split); }
    const bool fresh = !VER || sp == c0;
    const bool none = VER && j_lo >= j_hi;                              // no row of the tile has keys in this chunk
    const int s0 = j_lo / SK, nsteps = j_lo < j_hi ? (j_hi - 1) / SK - s0 + 1 : 0;

    // Step loads: thread slot S = (wave*NLD + u)*64 + lane of a K (V) stage holds the 16-byte column
    // (S % SLOTS) ^ kswz(key) (vswz(key)) of key row key = S / SLOTS, at a fixed byte offset from the step's first key
    // row. With a power of two of rows per wave, slot u's key is a bitwise or of the row of slot 0 and u * RPL, so its
    // swizzle is that of slot 0 XOR a constant: two registers hold a wave's offsets instead of 2 NLD.
    const unsigned krow_b = (unsigned)(krow * sizeof(KE));
    constexpr int RPL = 64 / SLOTS;                      // key rows of one 64-slot load
    constexpr bool XORU = ((NLD * RPL) & (NLD * RPL - 1)) == 0 && Cf::NLR % Cf::NW == 0;
    unsigned ld_koff[XORU ? 1 : NLD], ld_voff[XORU ? 1 : NLD];
#pragma unroll
    for (int u = 0; u < (XORU ? 1 : NLD); u++) {
        const int S = (wave * NLD + u) * 64 + lane, key = S / SLOTS;
        ld_koff[u] = (unsigned)(((S % SLOTS) ^ kswz(key)) * 8 * sizeof(KE)) + (XORU ? 0u : (unsigned)key * krow_b);
        ld_voff[u] = (unsigned)(((S % SLOTS) ^ vswz(key)) * 8 * sizeof(KE)) + (XORU ? 0u : (unsigned)key * krow_b);
    }
    const unsigned ld_row = XORU ? (unsigned)(wave * NLD * RPL + lane / SLOTS) * krow_b : 0u;
    auto k_off = [&](int u) -> unsigned {
        if constexpr (XORU) return (ld_koff[0] ^ (unsigned)(kswz(u * RPL) * 8 * sizeof(KE))) + u * RPL * krow_b;
        else return ld_koff[u];
    };
    auto v_off = [&](int u) -> unsigned {
        if constexpr (XORU) return (ld_voff[0] ^ (unsigned)(vswz(u * RPL) * 8 * sizeof(KE))) + u * RPL * krow_b;
        else return ld_voff[u];
    };
    // Step k of the walk goes into stage k % 2.
    // 16-bit caches: buffer loads straight into LDS over the byte range the workgroup may read (the keys below
    // hi_b, or a ring that they fill), so the rows past the last key of a step read as zeros (they are masked) without clamping.
    // (Verify runs hold to the keys [j_lo, j_hi) of the chunk on both sides: a ring may end before it was ever filled, and a
    // cache may be filled from the window on only. Rows below the range get offsets below zero, which are out of range too.)
    // fp32 caches: rows past the last key re-read that row, so every load is in bounds.
    // Byte offsets have 32 bits. FAR: the range is that of one step, at a 64-bit address. Otherwise one range from the start of
    // the sequence serves every step (host: below 4 GiB): forming it per step cost prompts 1-3% (T = 1024 of 16 q-heads over 8
    // 26.1 -> 26.9 us), verify runs nothing (16 trees of 8 nodes 129.4 -> 128.1 us).
    const int kv_rows = max(1, p.kv_cap > 0 ? min(p.kv_cap, hi_b) : hi_b);
    const uint32_t kv_bytes = FAR ? 0u : (uint32_t)(kv_rows - 1) * krow_b + (uint32_t)(HD * sizeof(KE));
    const __amdgpu_buffer_rsrc_t krs = make_rsrc(Kb, kv_bytes), vrs = make_rsrc(Vb, kv_bytes);      // !FAR
    int it_cur = 0;                                                     // the step being computed
    // Step k < 0 is a no-op step: every lane is out of range, so its loads write zeros into the stage of the step
    // before (already consumed by every wave) and touch no memory; this keeps the issue points branch-free.
    // step_ld forms a step's range (FAR: rows r0 .. of the step, below key hi), first byte offset and stages; issue_part issues
    // slots [u0, u1) of the thread's NLD (K and V each).
    struct StepLd { unsigned char *kd, *vd; const char *k, *v; uint32_t bytes, soff; int s; };
    auto step_ld = [&](int s, int stage, bool real, int r0, int hi) {
        StepLd st;
        st.s = s;
        st.kd = smem + (size_t)stage * Cf::STAGE;
        st.vd = st.kd + Cf::HALF;
        if constexpr (FAR) {
            const size_t off = (size_t)(unsigned)__builtin_amdgcn_readfirstlane(key_row(p, s * SK) + r0) * krow_b;
            const int rows = min(SK, hi - s * SK) - r0;
            st.k = reinterpret_cast<const char *>(Kb) + off;
            st.v = reinterpret_cast<const char *>(Vb) + off;
            st.bytes = real && rows > 0 ? (uint32_t)(rows - 1) * krow_b + (uint32_t)(HD * sizeof(KE)) : 0u;
            st.soff = 0u - (uint32_t)r0 * krow_b;
        } else {
            // (the range check covers the vector offset, which holds the step's offset too)
            st.soff = !real ? kv_bytes : (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned)key_row(p, s * SK) * krow_b));
        }
        return st;
    };
    auto prep = [&](int k) {
        const int kst = k < 0 ? it_cur + 1 : k;
        return step_ld(s0 + kst, kst % 2, k >= 0, 0, VER ? j_hi : hi_b);
    };
    auto issue_part = [&](const StepLd &st, int u0, int u1) {
        unsigned row = ld_row + st.soff;
        if constexpr (FAR) asm volatile("" : "+v"(row));                // offsets formed here, not held across the step loop
#pragma unroll
        for (int u = 0; u < NLD; u++) {
            if (u < u0 || u >= u1) continue;
            const int i = wave * NLD + u;
            if (Cf::NLR % Cf::NW != 0 && i >= Cf::NLR) continue;       // wave-uniform: past the tile
            unsigned koff = k_off(u) + row, voff = v_off(u) + row;
            if constexpr (!DMA) {
                if (FAR ? st.bytes == 0 : st.soff >= kv_bytes) continue;
                const int S = i * 64 + lane;
                if (st.s * SK + SK > hi_b) {
                    const unsigned key = (unsigned)(S / SLOTS), lim = (unsigned)(hi_b - 1 - st.s * SK);
                    if (key > lim) { koff -= (key - lim) * krow_b; voff -= (key - lim) * krow_b; }
                }
                const char *kp = FAR ? st.k : reinterpret_cast<const char *>(Kb), *vp = FAR ? st.v : reinterpret_cast<const char *>(Vb);
                *reinterpret_cast<u32x4 *>(st.kd + (size_t)S * 16) = load8_op<KVT, F16>(reinterpret_cast<const KE *>(kp + koff));
                *reinterpret_cast<u32x4 *>(st.vd + (size_t)S * 16) = load8_op<KVT, F16>(reinterpret_cast<const KE *>(vp + voff));
            } else if constexpr (FAR) {
                buffer_load_lds16<VER>(make_rsrc(st.k, st.bytes), st.kd + (size_t)i * 1024, (int)koff);
                buffer_load_lds16<VER>(make_rsrc(st.v, st.bytes), st.vd + (size_t)i * 1024, (int)voff);
            } else {
                buffer_load_lds16(krs, st.kd + (size_t)i * 1024, (int)koff);
                buffer_load_lds16(vrs, st.vd + (size_t)i * 1024, (int)voff);
            }
        }
    };
    auto issue = [&](int k) { issue_part(prep(k), 0, NLD); };
    // The next step's loads go out in four parts spread over the current step (between the QK batches, after
    // the softmax, between the PV batches): a workgroup's 8 waves issuing all of them at once stalled every wave
    // on the vector memory pipe for about a thousand cycles per step. (Verify runs wait for HBM, not for the pipe: all at
    // once, at the start.)
    constexpr int NPART = 4, PPART = (NLD + NPART - 1) / NPART;
    auto issue_pt = [&](const StepLd &st, int pt) {
        if (VER) { if (pt == 0) issue_part(st, 0, NLD); }
        else issue_part(st, pt * PPART, min(NLD, (pt + 1) * PPART));
    };
    if (nsteps > 0 && fresh) issue_part(step_ld(s0, 0, true, VER ? j_lo % SK : 0, VER ? j_hi : hi_b), 0, NLD);

    // The Q tile goes through LDS as well (16 bytes per lane of whole rows, where fragment loads straight from memory
    // touch 64 bytes of 16 rows each), in the stage that step 1 will fill, in the K layout: 16-byte column c of tile row R
    // in slot c ^ kswz(R), rows past the last as zeros. Row rho of a half tile is token rho / GRP, head rho % GRP.
    unsigned char *qs = smem + Cf::STAGE;
    auto tok_of = [&](int rho) { return (int)((unsigned)(rho * a.grp_mul) >> 16); };    // rho / GRP
    if (fresh) {
        constexpr bool QDMA = QT != DT_FP32;
        f32x4 raw[QDMA ? 1 : Cf::NQL][2];
#pragma unroll
        for (int u = 0; u < Cf::NQL; u++) {
            const int i = wave * Cf::NQL + u, hb = pair && i * RPL >= HR ? 1 : 0;
            const int R = i * RPL + lane / SLOTS, rho = R - hb * HR, nr = (tok1[hb] - tok0[hb]) * GRP;
            const int off = (rho + tok_of(rho) * (p.NQ - GRP)) * HD + ((lane % SLOTS) ^ kswz(R)) * 8;
            const QE *qb = reinterpret_cast<const QE *>(p.Q) + ((size_t)(seq * p.T + tok0[hb]) * p.NQ + kvh * GRP) * HD;
            if (QDMA && !a.q_al) {                                      // Q off a 16-byte boundary: through registers
                u32x4 v = u32x4{0u, 0u, 0u, 0u};
                if (rho < nr) v = *reinterpret_cast<const u32x4 *>(qb + off);
                *reinterpret_cast<u32x4 *>(qs + (size_t)i * 1024 + lane * 16) = v;
            } else if constexpr (QDMA) {
                const __amdgpu_buffer_rsrc_t qr = make_rsrc(qb, (uint32_t)((nr + tok_of(max(nr - 1, 0)) * (p.NQ - GRP)) * HD * 2));
                buffer_load_lds16(qr, qs + (size_t)i * 1024, rho < nr ? off * 2 : -16);
            } else {
                raw[u][0] = raw[u][1] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (rho < nr) {
                    raw[u][0] = *reinterpret_cast<const f32x4 *>(qb + off);
                    raw[u][1] = *reinterpret_cast<const f32x4 *>(qb + off + 4);
                }
            }
        }
        if constexpr (!QDMA)
#pragma unroll
            for (int u = 0; u < Cf::NQL; u++) {
                const f32x4 x = raw[u][0], y = raw[u][1];
                *reinterpret_cast<u32x4 *>(qs + (size_t)(wave * Cf::NQL + u) * 1024 + lane * 16) =
                    u32x4{pack2<F16>(x.x, x.y), pack2<F16>(x.z, x.w), pack2<F16>(y.x, y.y), pack2<F16>(y.z, y.w)};
            }
    }
    // This wave's row blocks: block rb covers rows [lrow[rb], lrow[rb] + 16) of half tile hb. Positions per row (an invalid
    // row has pos = -1 and attends nothing), and the wave-uniform key span of each block (positions grow with the row's
    // token).
    const int hb = pair ? rg * RB * 16 / HR : 0;
    const int htok = tok0[hb], hrows = (tok1[hb] - tok0[hb]) * GRP;
    int lrow[RB], rpos[RB];
    uint32_t anc[RB];                                                   // verify: tree masks of the rows (relative to pbase)
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        lrow[rb] = rg * RB * 16 + rb * 16 - hb * HR;
        rpos[rb] = lrow[rb] + ln < hrows ? pbase + htok + tok_of(lrow[rb] + ln) : -1;
        if constexpr (VER) anc[rb] = p.anc && rpos[rb] >= 0 ? p.anc[(size_t)seq * p.T + rpos[rb] - pbase] : 0u;
    }
    int wlo[RB], whi[RB], lo_max[RB], pos_min[RB];
    int wlo_all = INT_MAX, whi_all = -1;
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        const int rho1 = min(hrows, lrow[rb] + 16);
        wlo[rb] = INT_MAX; whi[rb] = -1; lo_max[rb] = 0; pos_min[rb] = INT_MAX;
        if (lrow[rb] < rho1) {
            const int pf = pbase + htok + tok_of(lrow[rb]), pl = pbase + htok + tok_of(rho1 - 1);
            wlo[rb] = max(win_lo(pf, p.window), j_lo); whi[rb] = min(pl, j_hi - 1);
            lo_max[rb] = win_lo(pl, p.window); pos_min[rb] = VER && p.anc ? pbase - 1 : pf;   // tree keys: per key
        }
        wlo_all = min(wlo_all, wlo[rb]); whi_all = max(whi_all, whi[rb]);
    }

    float m[RB], l[RB];
    f32x4 acc[RB][DB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        m[rb] = kNegInf; l[rb] = 0.f;
#pragma unroll
        for (int db = 0; db < DB; db++) {
            acc[rb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
            asm volatile("" : "+v"(acc[rb][db]));                       // cleared here, under the loads, not after the wait
        }
    }
    // Q fragments: lane (row ln, group g) holds dims 32 ks + 8 g .. of its rows.
    if (fresh) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
                qop[rb][ks] = *reinterpret_cast<const u32x4 *>(qs + (rg * RB * 16 + rb * 16 + ln) * ROWB + (((4 * ks + g) ^ kswz(ln)) << 4));
    }

    // Per-lane LDS byte addresses inside a step stage (the key group's rows start at kg*KT). A slot index
    // occupies address bits 4.., and the row base has those bits clear, so "slot s ^ x" is an XOR on the
    // address: K fragment (ks, g) of row ln is at kaddr ^ (64 ks); V transpose-read block db of row
    // 4g + ln/4 is at vaddr ^ (32 db).
    const unsigned lds0 = (unsigned)(uintptr_t)smem;
    const int vr = 4 * g + (ln >> 2);
    const unsigned kaddr = lds0 + (kg * Cf::KT + ln) * ROWB + ((g ^ kswz(ln)) << 4);
    const unsigned vaddr = lds0 + Cf::HALF + (kg * Cf::KT + vr) * ROWB + 8 * (ln & 1) + ((((ln & 3) >> 1) ^ vswz(vr)) << 4);

    // One step's work for this wave's row blocks: qk_softmax, then pv. QK: the K fragments of a sub-tile are read in batches (inline asm,
    // one wait per batch, so the reads are not serialised behind the MFMAs) and every row block runs its MFMA chain on
    // them. Then one softmax update, then PV with V^T fragments in batches of transpose reads. A row that attends none
    // of the step's keys keeps its state exactly. Each issues half of the next step's loads.
    PFrag<F16> pop[NSUB][RB];
    auto qk_softmax = [&](int it, const StepLd &nxt) {
        int pt = 0;
        const int jw = (s0 + it) * SK + kg * Cf::KT;
        // Per-lane LDS bases, made opaque so that the XOR-swizzled fragment addresses are formed next to their
        // reads instead of being hoisted out of the step loop (which held ~30 address registers live and spilled).
        unsigned kbase = kaddr + (it & 1) * Cf::STAGE;
        asm volatile("" : "+v"(kbase));
        constexpr int NCH = NSUB == 1 ? 2 : 1;                          // independent MFMA chains per S fragment
        f32x4 s[NSUB][RB][NCH];
#pragma unroll
        for (int sub = 0; sub < NSUB; sub++)
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int ch = 0; ch < NCH; ch++) s[sub][rb][ch] = f32x4{0.f, 0.f, 0.f, 0.f};
        {
            // Software-pipelined: batch b = KPB k-steps of every sub-tile; QD batches are read ahead of their MFMAs, so
            // the LDS latency hides under them. The swizzle XORs the low four bits of a row's slot index, so the four
            // k-steps that differ there take an XOR of the base and the others an immediate offset.
            constexpr int KPB = RB == 1 ? 2 : 1, NB = KS / KPB, RPB = KPB * NSUB, QD = 2, NHI = KS / 4;
            auto ks_of = [](int o) { return (o % NHI) * 4 + o / NHI; };     // k-steps in reading order
            u32x4 kb[QD][RPB];
            auto rd = [&](auto b_c) {
                constexpr int b = decltype(b_c)::value;
                static_for<KPB>([&](auto kk_c) {
                    constexpr int kk = decltype(kk_c)::value, o = b * KPB + kk;
                    const unsigned kx = kbase ^ (64u * (o / NHI));
                    static_for<NSUB>([&](auto sub_c) {
                        constexpr int sub = decltype(sub_c)::value;
                        lds_read16<256 * (o % NHI) + sub * 16 * ROWB>(kb[b % QD][sub * KPB + kk], kx);
                    });
                });
            };
            static_for<QD - 1>([&](auto b_c) { rd(b_c); });
            static_for<NB>([&](auto b_c) {
                constexpr int b = decltype(b_c)::value, ahead = b + QD - 1 < NB ? QD - 1 : NB - 1 - b;
                if constexpr (b + QD - 1 < NB) rd(std::integral_constant<int, b + QD - 1>{});
                lds_wait<ahead * RPB>(kb[b % QD]);
                if (b == 0 || b == NB / 2) issue_pt(nxt, pt++);
#pragma unroll
                for (int kk = 0; kk < KPB; kk++)
#pragma unroll
                    for (int sub = 0; sub < NSUB; sub++)
#pragma unroll
                        for (int rb = 0; rb < RB; rb++)
                            s[sub][rb][kk % NCH] = mfma16<F16>(kb[b % QD][sub * KPB + kk], qop[rb][ks_of(b * KPB + kk)], s[sub][rb][kk % NCH]);
            });
        }
        float tv[NSUB][RB][4], mnew[RB];
        bool need = false;
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const bool full = jw >= j_lo && jw + Cf::KT <= j_hi && jw >= lo_max[rb] && jw + Cf::KT - 1 <= pos_min[rb];
            float mx = kNegInf;
#pragma unroll
            for (int sub = 0; sub < NSUB; sub++) {
                f32x4 sc = s[sub][rb][0];
                if constexpr (NCH == 2) sc += s[sub][rb][1];
                sc *= a.sl2;
#pragma unroll
                for (int i = 0; i < 4; i++) tv[sub][rb][i] = sc[i];
            }
            if (!full) {                                        // one wave-uniform test; per key only off the fast path
                const int kl = max(j_lo, win_lo(rpos[rb], p.window)) - jw - 4 * g, kh = min(j_hi - 1, rpos[rb]) - jw - 4 * g;
#pragma unroll
                for (int sub = 0; sub < NSUB; sub++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if ((16 * sub + i < kl) | (16 * sub + i > kh)) tv[sub][rb][i] = kNegInf;
                if (VER && p.anc) {
                    const int d0 = jw + 4 * g - pbase;
#pragma unroll
                    for (int sub = 0; sub < NSUB; sub++)
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const int d = d0 + 16 * sub + i;
                            if ((d >= 0) & ((d >= 32) | !((anc[rb] >> (d & 31)) & 1u))) tv[sub][rb][i] = kNegInf;
                        }
                }
            }
#pragma unroll
            for (int sub = 0; sub < NSUB; sub++)
#pragma unroll
                for (int i = 0; i < 4; i++) mx = fmaxf(mx, tv[sub][rb][i]);
            mx = max_over_groups(mx);
            mnew[rb] = mx > m[rb] + kRescaleThreshold ? mx : m[rb];
            need |= mnew[rb] != m[rb];
        }
        if (__any(need)) {
            // every block (an unmoved one has alpha = 1): a per-block condition here made the compiler keep two copies
            // of the accumulator
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                const float alpha = (mnew[rb] == m[rb]) ? 1.f : fast_exp2(m[rb] - mnew[rb]);
                l[rb] *= alpha; m[rb] = mnew[rb];
#pragma unroll
                for (int db = 0; db < DB; db++) acc[rb][db] *= alpha;
            }
        }
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const float mr = m[rb] == kNegInf ? 0.f : m[rb];    // no key seen yet: every score is -inf, exp2 gives 0
#pragma unroll
            for (int sub = 0; sub < NSUB; sub++) {
                float pv[4];
#pragma unroll
                for (int i = 0; i < 4; i++) pv[i] = fast_exp2(tv[sub][rb][i] - mr);
                l[rb] += (pv[0] + pv[1]) + (pv[2] + pv[3]);
                pop[sub][rb] = p_frag<F16>(pv[0], pv[1], pv[2], pv[3]);
            }
        }
    };
    auto pv = [&](int it, const StepLd &nxt) {
        int pt = NPART / 2;
        unsigned vbase = vaddr + (it & 1) * Cf::STAGE;
        asm volatile("" : "+v"(vbase));
        // PV with V^T fragments in batches of PB dim blocks, software-pipelined: batch b+1 is read before batch b's MFMAs.
        // As for K, the eight dim blocks that differ in the swizzled bits take an XOR of the base, the others (16-byte
        // slots 16 apart) an immediate offset.
        // NSUB == 2: PV on 16x16x32 over both sub-tiles at once (the order of keys inside an MFMA's reduction is free):
        // k-group g of the MFMA holds keys 4g..4g+3 of sub-tile 0 and then of sub-tile 1, which is what the lane's two
        // S^T fragments hold (B operand = the two P^T halves) and what two transpose reads of V give (A operand).
        constexpr int PB = RB == 1 ? 4 : 2, NPB = DB / PB, NHV = DB / 8;
        auto db_of = [](int o) { return (o % NHV) * 8 + o / NHV; };         // dim blocks in reading order
        u32x2 vb2[2][NSUB * PB];
        auto rdv = [&](auto b_c) {
            constexpr int b = decltype(b_c)::value;
            static_for<PB>([&](auto j_c) {
                constexpr int j = decltype(j_c)::value, o = b * PB + j;
                const unsigned vx = vbase ^ (32u * (o / NHV));
                static_for<NSUB>([&](auto sub_c) {
                    constexpr int sub = decltype(sub_c)::value;
                    lds_read_tr<256 * (o % NHV) + sub * 16 * ROWB>(vb2[b & 1][NSUB * j + sub], vx);
                });
            });
        };
        rdv(std::integral_constant<int, 0>{});
        static_for<NPB>([&](auto b_c) {
            constexpr int b = decltype(b_c)::value;
            u32x2 (&cur)[NSUB * PB] = vb2[b & 1];
            if constexpr (b + 1 < NPB) rdv(std::integral_constant<int, b + 1>{});
            lds_wait<(b + 1 < NPB) ? NSUB * PB : 0>(cur);
            if constexpr (NSUB == 2) {
#pragma unroll
                for (int j = 0; j < PB; j++)
#pragma unroll
                    for (int rb = 0; rb < RB; rb++) {
                        f32x4 &c = acc[rb][db_of(b * PB + j)];
                        c = mfma_pv32_hi<F16>(u32x4{cur[2 * j][0], cur[2 * j][1], cur[2 * j + 1][0], cur[2 * j + 1][1]},
                                              pop[0][rb], pop[1][rb], c);
                    }
#pragma unroll
                for (int j = 0; j < PB; j++)
#pragma unroll
                    for (int rb = 0; rb < RB; rb++) {
                        f32x4 &c = acc[rb][db_of(b * PB + j)];
                        c = mfma_pv32_lo<F16>(u32x4{cur[2 * j][0], cur[2 * j][1], cur[2 * j + 1][0], cur[2 * j + 1][1]},
                                              pop[0][rb], pop[1][rb], c);
                    }
            } else {
#pragma unroll
                for (int j = 0; j < PB; j++) {
                    f32x4 &c = acc[0][db_of(b * PB + j)];
                    c = mfma_pv16<F16, KVT != DT_FP32>(cur[j], pop[0][0], c);
                }
            }
            if (b == 0 || b == NPB / 2) issue_pt(nxt, pt++);
        });
    };

    // The wave's keys of step it start at jw(it) = (s0 + it) * SK + kg * KT. It attends steps [it0, it1]: before
    // and after them it only keeps the barriers and the loads going. Three loops instead of a skip branch keep the
    // step loop a single path (a skip path made the register allocator copy the accumulator on every step).
    auto fdiv = [](int x, int y) { return x >= 0 ? x / y : -((-x + y - 1) / y); };
    const int jb = s0 * SK + kg * Cf::KT;
    const int it0 = __builtin_amdgcn_readfirstlane(max(0, -fdiv(-(wlo_all - Cf::KT + 1 - jb), SK)));
    const int it1 = __builtin_amdgcn_readfirstlane(whi_all < 0 ? -1 : min(nsteps - 1, fdiv(whi_all - jb, SK)));
    auto sync_step = [&](int it) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                // this wave's loads of step it have landed
        __syncthreads();                                                // everyone's have, and step it-1 is consumed
        it_cur = it;
        return it + 1 < nsteps ? it + 1 : -1;
    };
    int it = 0;
    for (; it < min(it0, nsteps); it++) issue(sync_step(it));
    for (; it <= it1; it++) {
        const StepLd nxt = prep(sync_step(it));
        qk_softmax(it, nxt);
        pv(it, nxt);
    }
    for (; it < nsteps; it++) issue(sync_step(it));
    // The no-op loads of the last steps still write (zeros) into a stage: drain them before the merge reuses the
    // tile region for its exchange and statistics.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int rb = 0; rb < RB; rb++) l[rb] = sum_over_groups(l[rb]);
    __syncthreads();                                                 // every wave is done with the K/V tiles
    if (VER && sp + 1 < c1) {
        const int lo = max(win_lo(pbase + tok0[0], p.window), (sp + 1) * a.kv_split), hi = min(hi_b, (sp + 2) * a.kv_split);
        issue_part(step_ld(lo / SK, 0, true, lo % SK, hi), 0, NLD);
    }
    if (none) return;

    // Merge the KG key-group states of each row (waves kg = 0..KG-1 of a row group hold the same rows). Key group kg owns
    // output dim blocks [kg*DO, (kg+1)*DO): every wave publishes its rows' (m, l) and parks the other groups' blocks of its
    // accumulator in LDS; after one barrier every lane derives M = max m and L = sum l 2^(m - M) (key groups in order) and
    // sums its own blocks over the key groups in order 0..KG-1 (the same order for every row and tiling), each scaled by
    // 2^(m - M) / L (2^(m - M) for a split partial).
    // Verify runs: the merge's addresses are formed again for every chunk; hoisted out of the chunk loop they were held (spilled,
    // at HD 128) through the steps (16 sequences x 10 tokens of 16 q-heads over 4 of 128, 256-key chunks: 42.5 -> 41.0 us).
    int lm = ln, gm = g;
    if constexpr (VER) asm volatile("" : "+v"(lm), "+v"(gm));
    const int NQ = p.NQ;
    if (gm == 0) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) { stm[wave * RB * 16 + rb * 16 + lm] = m[rb]; stl[wave * RB * 16 + rb * 16 + lm] = l[rb]; }
    }
    float *xb = reinterpret_cast<float *>(xmem);                        // exchange (reuses the tiles)
    auto xslot = [&](int rb, int owner, int sender) {
        return xb + ((((size_t)(rb * RG + rg) * KG + owner) * (KG - 1) + (sender < owner ? sender : sender - 1)) * 16 + lm) * Cf::XSTR + 4 * gm;
    };
    // park the blocks of the other owners (constant indices keep acc in registers)
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
        static_for<KG>([&](auto o_c) {
            constexpr int O = decltype(o_c)::value;
            if (O == kg) return;
            float *dst = xslot(rb, O, kg);
#pragma unroll
            for (int j = 0; j < DO; j++) *reinterpret_cast<f32x4 *>(dst + 16 * j) = acc[rb][O * DO + j];
        });
    __syncthreads();
    float f[RB][KG];                                                    // the key groups' factors
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        float M = kNegInf, mk[KG];
#pragma unroll
        for (int k = 0; k < KG; k++) { mk[k] = stm[(rg * KG + k) * RB * 16 + rb * 16 + lm]; M = fmaxf(M, mk[k]); }
        float L = 0.f;
#pragma unroll
        for (int k = 0; k < KG; k++) {
            f[rb][k] = mk[k] == kNegInf ? 0.f : fast_exp2(mk[k] - M);
            if (mk[k] != kNegInf) L += stl[(rg * KG + k) * RB * 16 + rb * 16 + lm] * f[rb][k];
        }
        if (!split) {
            const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
            for (int k = 0; k < KG; k++) f[rb][k] *= inv;
        }
        const int rho = lrow[rb] + lm;
        if (kg == 0 && gm == 0 && rho < hrows) {
            const int t = tok_of(rho), r = seq * p.T + htok + t, h = kvh * GRP + rho - t * GRP;
            if (split) {
                const size_t pi = ((size_t)r * NQ + h) * a.part.ns_cap + sp;
                a.part.m[pi] = M; a.part.l[pi] = L;
            } else if (p.lse) {
                p.lse[(size_t)r * NQ + h] = (L > 0.f) ? (M + log2f(L)) * kLn2 : kNegInf;
            }
        }
    }
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        const int rho = lrow[rb] + lm;
        if (rho >= hrows) continue;
        const int t = tok_of(rho);
        const size_t ro = (size_t)(seq * p.T + htok + t) * NQ + kvh * GRP + rho - t * GRP;     // output row
        static_for<KG>([&](auto o_c) {
            constexpr int O = decltype(o_c)::value;
            if (O != kg) return;
#pragma unroll
            for (int j = 0; j < DO; j++) {
                f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < KG; k++) {
                    const f32x4 x = (k == O ? acc[rb][O * DO + j] : *reinterpret_cast<const f32x4 *>(xslot(rb, O, k) + 16 * j)) * f[rb][k];
                    o = k == 0 ? x : o + x;
                }
                const int d = 16 * (O * DO + j) + 4 * gm;
                if (split) {
                    *reinterpret_cast<f32x4 *>(a.part.acc + (ro * a.part.ns_cap + sp) * HD + d) = o;
                } else if constexpr (OT == DT_FP32) {
                    *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(p.O) + ro * HD + d) = o;
                } else {
                    const u32x2 wv = u32x2{pack2<OT == DT_F16>(o.x, o.y), pack2<OT == DT_F16>(o.z, o.w)};
                    *reinterpret_cast<u32x2 *>(reinterpret_cast<uint16_t *>(p.O) + ro * HD + d) = wv;
                }
            }
        });
    }
}

template <int HD, int RB, int RG, int KG_, int NSUB, int WPE, int KVT, int QT, int OT, bool VER, bool FAR>
__global__ void __launch_bounds__(RG * KG_ * 64) __attribute__((amdgpu_waves_per_eu(WPE)))
prefill_kernel(const PrefArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const Problem &p = a.p;
    int seq, kvh, qi;                                                   // sequence, KV head, tile from the last
    if constexpr (VER) {
        // Verify: runs of key chunks, KV heads and tiles of one run side by side.
        const int per = p.NKV * a.nht, it = (int)blockIdx.x / per, x = (int)blockIdx.x - it * per;
        int p0, c0, c_end, left;
        if (!find_run(p, a.kv_split, a.split_m, it, a.slots, seq, p0, c0, c_end, left)) return;
        qi = x / p.NKV; kvh = x - qi * p.NKV;
        for (;;) {
            seq = __builtin_amdgcn_readfirstlane(seq); c0 = __builtin_amdgcn_readfirstlane(c0);
            p0 = __builtin_amdgcn_readfirstlane(p0);
            const int c1 = __builtin_amdgcn_readfirstlane(min(c_end, c0 + left));
            u32x4 qop[RB][HD / 32];
            for (int sp = c0; sp < c1; sp++) prefill_item<HD, RB, RG, KG_, NSUB, KVT, QT, OT, true, FAR>(a, seq, p0, kvh, qi, sp, c0, c1, qop, smem);
            left -= c1 - c0;
            if (left <= 0) return;
            int n;
            do {                                                        // the next sequence with keys
                if (++seq >= p.nseq) return;                            // (unreachable while the counts agree)
                seq_chunks(p, a.kv_split, a.split_m, seq, p0, c0, n);
            } while (n <= 0);
            c_end = c0 + n;
            __syncthreads();                                            // every wave is done with the merge's LDS
        }
    } else {
        // XCD-aware work index: dispatch slot b runs on XCD b % 8, and the work items of one KV head (longest first) share
        // an XCD, so that head's K/V stays in one L2. Fewer heads than XCDs: a head's items are dealt in turn to its
        // `ways` XCDs; a multiple of 8 heads: an XCD takes its heads' items in turn; other counts: every head's longest
        // items first, over all XCDs. Long items of every head start first in each case: with the longest half of a head on
        // one XCD and the shortest on another, the 1377-token prompt of 24 q-heads over 4 KV heads took 75 instead of 56 us.
        // With a.fold the local slot k is folded: slots k and k + per/2 - which the dispatcher places on the same CU when
        // two workgroups fit a CU and the grid is one round - take the k-th longest and the k-th shortest item.
        const int per = (int)gridDim.x / 8, k_loc = (int)blockIdx.x / 8, h_loc = (per + 1) / 2, xcd = (int)blockIdx.x % 8;
        const int k_f = !a.fold || k_loc < h_loc ? k_loc : per - 1 - (k_loc - h_loc);
        int head, item;                                                     // head = sequence * NKV + KV head
        if (a.ways > 0) { head = xcd / a.ways; item = k_f * a.ways + xcd % a.ways; }
        else if (a.ways < 0) { item = k_f / -a.ways; head = xcd + 8 * (k_f + item * a.ways); }
        else { const int i = 8 * k_f + xcd; item = i / a.heads; head = i - item * a.heads; }
        if (item >= a.nitems || head >= a.heads) return;
        // (runtime divisions take ~200 cycles each: skipped where the launch makes them trivial)
        seq = p.nseq > 1 ? head / p.NKV : 0; kvh = head - seq * p.NKV;
        qi = a.nsplit > 1 ? item / a.nsplit : item;
        u32x4 qop[RB][HD / 32];
        prefill_item<HD, RB, RG, KG_, NSUB, KVT, QT, OT, false, FAR>(a, seq, 0, kvh, qi, item - qi * a.nsplit, 0, 0, qop, smem);
    }
}

// ---------------------------------------------------------------- host side
// Tile shapes: 8 waves (two per SIMD) as 4 row groups x 2 key groups, 16 rows and HD accumulator columns per wave, a
// 64-row workgroup tile, 64-key steps (two 16-key sub-tiles per wave) in two LDS stages. HD 512: 32-key steps (a 32-key
// stage of HD 512 is 64 KB) and a 16 x 512 accumulator per wave.
// HD 256 has two larger tiles for launches of more than one round of 64-row workgroups; all three share the step, the
// key groups and the merge order, so a row's bits do not depend on which one ran it.
//   W = 1: 12 waves (6 row groups, three per SIMD, 164 VGPRs), 96 rows.
//   W = 2: 8 waves of two 16-row blocks each (256 VGPRs), 128 rows: every K and V fragment read from LDS feeds two MFMAs,
//          so a row costs 18 ns per 64-key step against 22 ns at 64 rows (bf16).
// What bounds a step: MFMA issue and VALU issue add up on a SIMD (a probe with two waves per SIMD measures 16.5 cycles per
// 16x16x32 MFMA and about 2.2 more for every VALU op beside it), and a 128-row bf16 step holds 192 MFMAs (3170 cycles)
// and about 380 VALU ops per SIMD; it runs in about 5000 cycles. Neither the LDS (256 bytes per clock against 320 KB per
// step) nor the L2 stream (without the loads the 4096-token window prompt gains 3%) is near its limit, and letting the
// second wave of each SIMD run half a step behind the first, to put one's MFMAs under the other's softmax, changed nothing.
// WPE: waves per SIMD the register allocation must allow.
template <int HD, int W> struct PrefTile;
template <> struct PrefTile<128, 0> { static constexpr int RB = 1, RG = 4, KG = 2, NSUB = 2, WPE = 2; };
template <> struct PrefTile<256, 0> { static constexpr int RB = 1, RG = 4, KG = 2, NSUB = 2, WPE = 2; };
template <> struct PrefTile<256, 1> { static constexpr int RB = 1, RG = 6, KG = 2, NSUB = 2, WPE = 3; };
template <> struct PrefTile<256, 2> { static constexpr int RB = 2, RG = 4, KG = 2, NSUB = 2, WPE = 2; };
template <> struct PrefTile<512, 0> { static constexpr int RB = 1, RG = 4, KG = 2, NSUB = 1, WPE = 2; };
// W = 3: verify runs (also for 17-32 rows: a 32-row tile of four waves took 128 against 118 us for 12 sequences x 12 tokens
// of 16 q-heads over 8, for its slower K/V requests).
template <> struct PrefTile<128, 3> { static constexpr int RB = 1, RG = 4, KG = 2, NSUB = 2, WPE = 4; };
template <> struct PrefTile<256, 3> { static constexpr int RB = 1, RG = 4, KG = 2, NSUB = 2, WPE = 2; };
template <int HD, int W>
using PrefTileCfg = PrefCfg<HD, PrefTile<HD, W>::RB, PrefTile<HD, W>::RG, PrefTile<HD, W>::KG,
                            PrefTile<HD, W>::NSUB>;

template <int HD, int W, int KVT, int QT, int OT, bool VER = false, bool FAR = VER>
static hipError_t launch_pref_t(const PrefArgs &a, dim3 grid, hipStream_t st) {
    using T = PrefTile<HD, W>;
    using Cf = PrefTileCfg<HD, W>;
    static bool configured = false;
    auto kern = prefill_kernel<HD, T::RB, T::RG, T::KG, T::NSUB, T::WPE, KVT, QT, OT, VER, FAR>;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)Cf::lds(VER));
        if (e != hipSuccess) return e;
        configured = true;
    }
    hipLaunchKernelGGL(kern, grid, dim3(Cf::NT), Cf::lds(VER), st, a);
    return hipGetLastError();
}

// Whether a sequence's K (or V) rows, plus the largest offset inside a step past them, pass 32-bit byte offsets: the narrow
// tiles have a form that addresses each step in 64 bits.
static bool pref_far(const Problem &p) {
    const long long rows = p.kv_cap > 0 ? p.kv_cap : (long long)p.max_pos + 1;
    return (rows + 128) * p.NKV * p.HD * (p.kv_dtype == DT_FP32 ? 4 : 2) >= 1ll << 32;
}

template <int KVT, int QT, int OT>
static hipError_t pref_dispatch_hd(const PrefArgs &a, int wide, dim3 grid, hipStream_t st) {
    if (pref_far(a.p))
        return a.p.HD == 128 ? launch_pref_t<128, 0, KVT, QT, OT, false, true>(a, grid, st)
             : a.p.HD == 256 ? launch_pref_t<256, 0, KVT, QT, OT, false, true>(a, grid, st)
             : a.p.HD == 512 ? launch_pref_t<512, 0, KVT, QT, OT, false, true>(a, grid, st) : hipErrorInvalidValue;
    switch (a.p.HD) {
    case 128: return launch_pref_t<128, 0, KVT, QT, OT>(a, grid, st);
    case 256:
        if constexpr (KVT != DT_FP32) {
            if (wide == 1) return launch_pref_t<256, 1, KVT, QT, OT>(a, grid, st);
            if (wide == 2) return launch_pref_t<256, 2, KVT, QT, OT>(a, grid, st);
        }
        return launch_pref_t<256, 0, KVT, QT, OT>(a, grid, st);
    case 512: return launch_pref_t<512, 0, KVT, QT, OT>(a, grid, st);
    default: return hipErrorInvalidValue;
    }
}

// Per tile shape (head dim, W): rows of a half tile, workgroups resident per CU, keys per step, and the measured cost of
// a workgroup on bf16 caches in us: its start and end, a step with both half tiles at work, and a step with one.
struct PrefShape { int hr, per_cu, sk; float ov, full, half; };
template <int HD, int W> static PrefShape pref_shape_t(float ov, float full, float half) {
    using Cf = PrefTileCfg<HD, W>;
    return PrefShape{Cf::HR, (int)std::max<size_t>(1, (160u << 10) / Cf::LDS), Cf::SK, ov, full, half};
}
static PrefShape pref_shape(int HD, int wide) {
    switch (HD) {
    case 128: return pref_shape_t<128, 0>(4.5f, 0.8f, 0.6f);
    case 256:
        return wide == 2 ? pref_shape_t<256, 2>(9.f, 2.35f, 1.43f)
               : wide    ? pref_shape_t<256, 1>(7.f, 1.9f, 1.25f)
                         : pref_shape_t<256, 0>(5.5f, 1.45f, 1.05f);
    case 512: return pref_shape_t<512, 0>(8.f, 1.37f, 1.08f);
    default: return PrefShape{0, 1, 64, 0.f, 0.f, 0.f};
    }
}
static int pref_half_rows(int HD) { return pref_shape(HD, 0).hr; }
static int pref_per_cu(int HD) { return pref_shape(HD, 0).per_cu; }

size_t prefill_lds_bytes(int HD) {
    switch (HD) {
    case 128: return PrefTileCfg<128, 0>::LDS;
    case 256: return PrefTileCfg<256, 0>::LDS;
    case 512: return PrefTileCfg<512, 0>::LDS;
    default: return 0;
    }
}

int device_cus() {
    static std::atomic<int> cus[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int n = cus[dev].load(std::memory_order_relaxed);
    if (n == 0 && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess)
        cus[dev].store(n, std::memory_order_relaxed);
    return n;
}

// Key split for kv_split = -1: when the unsplit grid would fill at most half of the workgroup slots (a short run
// of queries over a long cached prefix), cut the keys into as many absolute splits as whole grids fit on them.
int prefill_auto_split(const Problem &p) {
    if (p.NQ % p.NKV) return 0;
    const int GRP = p.NQ / p.NKV, HR = pref_half_rows(p.HD);
    if (HR == 0 || GRP > HR) return 0;
    const int tqh = HR / GRP, nht = (p.T + tqh - 1) / tqh;
    const long nwg = (long)p.nseq * p.NKV * ((nht + 1) / 2);
    const long slots = (long)device_cus() * pref_per_cu(p.HD);
    if (nwg <= 0 || 2 * nwg > slots) return 0;
    const int nsplit = (int)(slots / nwg);
    const int keys = p.max_pos + 1;
    int ks = (keys + nsplit - 1) / nsplit;
    ks = ((ks + 63) / 64) * 64;
    return ks >= keys ? 0 : ks;
}

// How a launch is cut into work items: the tile shape, and one tile per item (a full one or, `one_half`, a half tile whose
// other waves only load) or a causal pair of half tiles.
struct PrefPlan { int wide, pair, tqh, nht; };
static PrefPlan pref_plan(const PrefShape &sh, int wide, int GRP, int T, bool pair, bool one_half) {
    const int tqh = (pair || one_half ? 1 : 2) * sh.hr / GRP;
    return PrefPlan{wide, pair ? 1 : 0, tqh, (T + tqh - 1) / tqh};
}
// Estimated time of a plan in us: the items, longest first, dealt in a snake over the slots (slot c takes items c, 2K-1-c,
// 2K+c, ...), which is about what longest-first dispatch gives; the longest of five slots counts.
static float pref_cost(const PrefShape &sh, const PrefPlan &pl, const Problem &p, int kv_split, int nsplit, int slots) {
    const int heads = p.nseq * p.NKV, base = std::max(0, p.max_pos - p.T + 1), GRP = p.NQ / p.NKV;
    const bool both = pl.pair || pl.tqh * GRP > sh.hr;
    auto cost = [&](long i) {
        const int r = (int)(i / heads / nsplit), t0 = (pl.nht - 1 - r) * pl.tqh, hi = base + std::min(p.T, t0 + pl.tqh);
        const int lo = p.window > 0 ? std::max(0, base + t0 - p.window + 1) : 0;
        int n = (hi - 1) / sh.sk - lo / sh.sk + 1;
        if (kv_split > 0) n = std::min(n, kv_split / sh.sk);
        if (!pl.pair) return sh.ov + n * (both ? sh.full : sh.half);
        const int s = std::min(n, r == pl.nht - 1 - r ? 0 : (base + (r + 1) * pl.tqh - 1) / sh.sk + 1);
        return sh.ov + s * sh.full + (n - s) * sh.half;
    };
    const long items = (long)heads * nsplit * (pl.pair ? (pl.nht + 1) / 2 : pl.nht), rounds = (items + slots - 1) / slots;
    const long every = std::max(1L, rounds / 16);                       // sampled rounds of a long launch
    float worst = 0.f;
    for (int k = 0; k < 5; k++) {
        const long c = (long)(slots - 1) * k / 4;
        float sum = 0.f;
        for (long r = 0; r < rounds; r += every) {
            const long i = r * slots + (r & 1 ? slots - 1 - c : c);
            if (i < items) sum += cost(i) * (float)std::min(every, rounds - r);
        }
        worst = std::max(worst, sum);
    }
    return worst;
}
// The plan of a launch. If half tiles of the narrow shape fit the device in one round, one each: the longest item then has
// the cheapest steps (a causal pair would only add the short half's). Otherwise the cheapest by pref_cost among the shapes
// (the larger ones on 16-bit caches: the fp32 cache's register staging spills in them) with one tile per item or, for
// causal prompts whose work varies (no window, prefix shorter than the chunk), pairs. Measured at bf16 unless said:
//   16 q-heads over 8 KV heads, T = 1024: pairs of 32 rows 25.7 us; 64-row tiles 29.6, 96-row pairs 30.7, 128-row pairs 35.1
//   the same, T = 4096, window 1024: 128-row tiles 101 us; 64-row 114, 96-row 117
//   24 over 4, T = 1377 (f16): 96-row tiles 42.4 us; 64-row tiles 50.1 and pairs 64.6, 128-row tiles 50.5, 96-row pairs 54.7
//   16 over 1 of 512, T = 1024: pairs 46.1 us, 64-row tiles 55.0
static PrefPlan choose_plan(const Problem &p, int kv_split, int nsplit, int ncu) {
    const int GRP = p.NQ / p.NKV;
    const PrefShape s0 = pref_shape(p.HD, 0);
    const PrefPlan small = pref_plan(s0, 0, GRP, p.T, false, true);
    const int slots0 = std::max(ncu, 1) * s0.per_cu;
    if ((long)p.nseq * p.NKV * nsplit * small.nht <= slots0) return small;
    const bool causal = kv_split == 0 && p.window == 0 && p.max_pos < 2 * p.T;
    PrefPlan best = pref_plan(s0, 0, GRP, p.T, causal, false);
    float cost = pref_cost(s0, best, p, kv_split, nsplit, slots0);
    auto consider = [&](const PrefShape &sh, const PrefPlan &pl) {
        const float c = pref_cost(sh, pl, p, kv_split, nsplit, std::max(ncu, 1) * sh.per_cu);
        if (c < cost) { cost = c; best = pl; }
    };
    if (causal) consider(s0, pref_plan(s0, 0, GRP, p.T, false, false));
    if (p.HD == 256 && p.kv_dtype != DT_FP32 && !pref_far(p))
        for (int w = 1; w <= 2; w++) {
            const PrefShape sh = pref_shape(256, w);
            consider(sh, pref_plan(sh, w, GRP, p.T, false, false));
            if (causal) consider(sh, pref_plan(sh, w, GRP, p.T, true, false));
        }
    return best;
}

hipError_t launch_prefill(const Problem &p, int kv_split, const Partials &part, hipStream_t st) {
    if (p.NQ % p.NKV || p.anc || p.pos_mode != 1) return hipErrorInvalidValue;
    const int GRP = p.NQ / p.NKV;
    if (pref_half_rows(p.HD) == 0 || GRP > pref_half_rows(p.HD)) return hipErrorInvalidValue;
    if (kv_split < 0 || (kv_split > 0 && kv_split % 64)) return hipErrorInvalidValue;
    const int nsplit = kv_split > 0 ? p.max_pos / kv_split + 1 : 1;
    if (kv_split > 0 && nsplit > part.ns_cap) return hipErrorInvalidValue;
    const int ncu = device_cus();
    const PrefPlan pl = choose_plan(p, kv_split, nsplit, ncu);
    const int wide = pl.wide, per_cu = pref_shape(p.HD, wide).per_cu, heads = p.nseq * p.NKV;
    const long nitems = (long)(pl.pair ? (pl.nht + 1) / 2 : pl.nht) * nsplit, nwg = heads * nitems;
    if (nwg <= 0 || nwg > (1L << 30)) return hipErrorInvalidConfiguration;
    const int fold = (per_cu >= 2 && nwg <= (long)per_cu * ncu) ? 1 : 0;
    const int ways = heads < 8 && 8 % heads == 0 ? 8 / heads : heads % 8 == 0 ? -(heads / 8) : 0;
    const long per = ways > 0 ? (nitems + ways - 1) / ways : (nwg + 7) / 8;
    PrefArgs a{p, part, kv_split, 0u, pl.nht, nsplit, pl.tqh, pl.pair, (int)nitems, heads, GRP, p.scale * kLog2e, fold,
               (reinterpret_cast<uintptr_t>(p.Q) & 15) == 0 ? 1 : 0, 65535 / GRP + 1, 0, ways};
    dim3 grid((unsigned)(8 * per));
    hipError_t e = hipErrorInvalidValue;
    const int kv = p.kv_dtype, q = p.q_dtype, o = p.o_dtype;
    if (kv == DT_F16 && q == DT_FP32 && o == DT_FP32) e = pref_dispatch_hd<DT_F16, DT_FP32, DT_FP32>(a, wide, grid, st);
    else if (kv == DT_BF16 && q == DT_FP32 && o == DT_FP32) e = pref_dispatch_hd<DT_BF16, DT_FP32, DT_FP32>(a, wide, grid, st);
    else if (kv == DT_FP32 && q == DT_FP32 && o == DT_FP32) e = pref_dispatch_hd<DT_FP32, DT_FP32, DT_FP32>(a, wide, grid, st);
    else if (kv == DT_F16 && q == DT_F16 && o == DT_F16) e = pref_dispatch_hd<DT_F16, DT_F16, DT_F16>(a, wide, grid, st);
    else if (kv == DT_BF16 && q == DT_BF16 && o == DT_BF16) e = pref_dispatch_hd<DT_BF16, DT_BF16, DT_BF16>(a, wide, grid, st);
    else return hipErrorInvalidValue;
    if (e != hipSuccess || kv_split <= 0) return e;
    return launch_combine(p, kv_split, part, st);
}

// Verify and tree runs (more than 16 rows per KV head): the keys in absolute chunks, found on the device from the positions
// (find_run), one partial per (row, chunk). Against a tile of four waves that each walk all 16-key tiles of the chunk, two
// key groups and 64-key steps halve the chain of a chunk: a 7-token draft over 3001 keys (24 workgroups) takes 24.3 instead
// of 47.0 us. 16 trees of 8 nodes over up to 16K keys (876 chunks, bound by HBM: 26 GB/s per CU inside the loop) take 128
// against 133 us; one chunk per workgroup there 134. 32-key steps took 158 us with two stages (a step then is one HBM
// latency) and 153 with four.
bool verify_tile_supported(const Problem &p, int chunk) {
    return (p.HD == 128 || p.HD == 256) && p.kv_dtype != DT_FP32 && (p.q_dtype == DT_FP32 || p.q_dtype == p.kv_dtype) &&
           p.NQ % p.NKV == 0 && p.NQ / p.NKV <= 2 * pref_half_rows(p.HD) && chunk > 0 && chunk % 32 == 0 &&
           (p.pos_mode == 1 || p.T == 1);
}

template <int KVT, int QT>
static hipError_t verify_dispatch(const PrefArgs &a, dim3 grid, hipStream_t st) {
    return a.p.HD == 128 ? launch_pref_t<128, 3, KVT, QT, DT_FP32, true>(a, grid, st)
                         : launch_pref_t<256, 3, KVT, QT, DT_FP32, true>(a, grid, st);
}

hipError_t launch_verify_tile(const Problem &p, int chunk, const Partials &part, hipStream_t st) {
    if (!verify_tile_supported(p, chunk)) return hipErrorNotSupported;
    if (p.max_pos / chunk + 1 > part.ns_cap) return hipErrorInvalidValue;
    const int GRP = p.NQ / p.NKV;
    const int tq = 64 / GRP, nt = (p.T + tq - 1) / tq;
    // Runs per (KV head, tile): as many as are resident at once, or of two to four rounds, where one leaves the device less
    // full. Their number bounds the grid: a workgroup without work still takes its LDS and reads the positions (about 1 us).
    const long long per = (long long)p.NKV * nt, res = std::max(1, device_cus()) * (p.HD == 128 ? 2 : 1);
    long long runs = 1;
    double use = 0.;
    for (int m = 1; m <= 4 && use < 0.9; m++) {
        const long long r = std::max(1ll, m * res / per), rounds = (r * per + res - 1) / res;
        const double u = (double)(r * per) / (double)(rounds * res);
        if (u > use) { use = u; runs = r; }
    }
    const long long wgs = std::min(chunk_items_bound(p, chunk), runs) * per;
    if (wgs > INT_MAX) return hipErrorInvalidConfiguration;
    Problem pr = p;
    if (p.pos_mode == 1) pr.pos_step = 0;                              // see seq_chunks
    PrefArgs a{pr, part, chunk, div_magic(chunk), nt, 1, tq, 0, 0, p.nseq * p.NKV, GRP, p.scale * kLog2e, 0,
               (reinterpret_cast<uintptr_t>(p.Q) & 15) == 0 ? 1 : 0, 65535 / GRP + 1,
               (int)runs, 0};
    const dim3 grid((unsigned)wgs);
    const bool q32 = p.q_dtype == DT_FP32;
    if (p.kv_dtype == DT_F16)
        return q32 ? verify_dispatch<DT_F16, DT_FP32>(a, grid, st) : verify_dispatch<DT_F16, DT_F16>(a, grid, st);
    return q32 ? verify_dispatch<DT_BF16, DT_FP32>(a, grid, st) : verify_dispatch<DT_BF16, DT_BF16>(a, grid, st);
}

}  // namespace dgx
