// Internal launch descriptors shared by the kernels and the C-ABI layer (not part of the public interface).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <climits>

namespace dgx {

// A batch of `nseq` sequences, each with `T` query tokens over its own KV cache (K/V at seq * kv_stride elements).
// Token (s, t) has global row index r = s * T + t (Q/O/LSE are [r][NQ][HD] / [r][NQ]).
// Its position is
//   pos_mode 0: pos_arr ? pos_arr[r] : base + r * pos_step              (launch_attn_decode_split rows)
//   pos_mode 1: (pos_arr ? pos_arr[s] : base) + t                        (a sequence of consecutive tokens)
// With anc, the tree of sequence s starts at tb = position of token (s, 0) and anc[r] masks keys >= tb.
struct Problem {
    const void *Q; int q_dtype;
    const void *K; const void *V; int kv_dtype;
    void *O; int o_dtype;
    float *lse;                       // optional [rows, NQ], natural log
    int nseq, T, NQ, NKV, HD;
    long kv_stride;
    int pos_mode, base, pos_step;
    const int *pos_arr;
    const uint32_t *anc;
    int max_pos;                      // host-side upper bound of every position (sizes the split grid)
    float scale;                      // resolved (> 0)
    int window;
    const void *const *Kp;            // optional device arrays of per-sequence K / V bases (override K, V + s*kv_stride)
    const void *const *Vp;
    const void *gate;                 // optional output gate [rows, NQ, HD]: O *= sigmoid(gate) (split path only)
    int gate_dtype;
    int kv_cap;                       // 0: key j in cache row j; > 0 (multiple of 64): ring buffer, row j % kv_cap
};

// Cache row of key j0, a multiple of 16: tiles of 16 (64 in prefill steps) keys never wrap inside a ring.
__device__ __forceinline__ int key_row(const Problem &p, int j0) {
    return p.kv_cap > 0 ? (int)((unsigned)j0 % (unsigned)p.kv_cap) : j0;
}

// K (v = false) or V cache base of sequence s.
template <class KE>
__device__ __forceinline__ const KE *kv_base(const Problem &p, bool v, int s) {
    const void *const *tab = v ? p.Vp : p.Kp;
    if (tab) return reinterpret_cast<const KE *>(tab[s]);
    return reinterpret_cast<const KE *>(v ? p.V : p.K) + (size_t)s * p.kv_stride;
}

// Split-KV partials in scratch: index (r * NQ + h) * ns_cap + c; m and l in the log2 domain (m = max of
// scale*log2(e)*q.k, l = sum of 2^(t - m)), acc = sum 2^(t - m) v, unnormalised.
struct Partials {
    float *m, *l, *acc;
    int ns_cap;
    // Set by launch_split when verify_kernel wrote the partials (seg_g > 0: its grid size and minimum run length;
    // the slots of a pair end at the first slot whose m is +inf); 0 for partials indexed by absolute key chunk.
    int seg_g = 0, seg_qmin = 0;
};

// Position of token t of sequence s, and the first key of its sliding window.
__device__ __forceinline__ int tok_pos(const Problem &p, int s, int t) {
    if (p.pos_mode == 0) {
        const int r = s * p.T + t;
        return p.pos_arr ? p.pos_arr[r] : p.base + r * p.pos_step;
    }
    return (p.pos_arr ? p.pos_arr[s] : p.base) + t;
}
__device__ __forceinline__ int win_lo(int pos, int window) {
    return (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
}

// x / C for 0 <= x < 2^31 and C >= 2, with M = div_magic(C): a runtime division costs a few hundred cycles on the path to a
// workgroup's first load. x M / 2^32 exceeds x / C by less than a half.
inline uint32_t div_magic(int C) { return (uint32_t)(0xffffffffu / (uint32_t)C) + 1u; }
__device__ __forceinline__ int div_by(int x, int C, uint32_t M) {
    const int q = (int)__umulhi((uint32_t)x, M);
    return q * C > x ? q - 1 : q;
}

// Inclusive prefix sum over the 64 lanes on the VALU (DPP row shifts and row broadcasts).
__device__ __forceinline__ int wave_scan64(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);     // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);     // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);     // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);     // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);     // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);     // row_bcast:31 into rows 2 and 3
    return v;
}

// Work item number `rest` -> (sequence, chunk c of C keys) and the key range [lo, hi) of the sequence's tokens,
// enumerating only the chunks that hold keys of them; called by whole waves with the same `rest`. M = div_magic(C). The
// workgroups with work come first in launch order and the dispatcher
// spreads them over all CUs; the tail of the upper-bound grid (false) exits at once. Two phases: first every chunk
// of each sequence but one, then that one: the shorter of its first and last chunk (both partial under a sliding
// window, only the last otherwise). The dispatcher hands workgroups out in
// index order and a CU that receives more workgroups than the others shares its bandwidth among them, so the short
// items go last, where they land on the CUs that get a third workgroup (measured: a CU with three full items runs
// 20% longer than one with two).
// The divisions by C are multiplications and the scans run on the VALU (2.2 -> about 1 us before a workgroup's first load).
// A form without the second pass over the positions took 57.9 against 57.5 us on the 564-workgroup decode batch, which is no
// more than runs of one build differ by; the two passes are the form that starts the short items no earlier than the others.
__device__ __forceinline__ bool find_item(const Problem &p, int C, uint32_t M, int rest, int &seq, int &c, int &lo, int &hi) {
    const int lane_ = threadIdx.x & 63, cmax = div_by(p.max_pos, C, M);
    seq = -1; c = 0;
    // Key range of sequence s's tokens, its first chunk and chunk count (positions ascend with the token).
    auto range = [&](int s, int &lo_s, int &hi_s, int &first, int &n) {
        const int p0 = tok_pos(p, s, 0), p1 = p.T > 1 ? tok_pos(p, s, p.T - 1) : p0;
        lo_s = win_lo(min(p0, p1), p.window); hi_s = max(p0, p1) + 1;
        if (p.pos_mode == 0)
            for (int t = 1; t + 1 < p.T; t++) {             // rows of their own positions
                const int ps = tok_pos(p, s, t);
                lo_s = min(lo_s, win_lo(ps, p.window)); hi_s = max(hi_s, ps + 1);
            }
        first = div_by(max(lo_s, 0), C, M);
        n = hi_s > 0 ? max(0, min(div_by(hi_s - 1, C, M), cmax) - first + 1) : 0;
    };
    // The phase-1 chunk of a sequence, counted from its first: the shorter of the first and the last.
    auto short_chunk = [&](int lo_s, int hi_s, int first, int n) {
        const int kf = min(hi_s, (first + 1) * C) - lo_s, kl = hi_s - max(lo_s, (first + n - 1) * C);
        return n >= 2 && kf >= kl ? n - 1 : 0;
    };
    for (int phase = 0; phase < 2; phase++) {
        for (int s0 = 0; s0 < p.nseq; s0 += 64) {
            int lo_s = 0, hi_s = 0, first = 0, n = 0;
            if (s0 + lane_ < p.nseq) range(s0 + lane_, lo_s, hi_s, first, n);
            const int m = phase == 0 ? max(n - 1, 0) : min(n, 1);   // items of this sequence in this phase
            const int sh = short_chunk(lo_s, hi_s, first, n), incl = wave_scan64(m);
            const unsigned long long hit = __ballot(incl > rest);
            if (hit) {
                const int l = __builtin_ctzll(hit), r = rest - (incl - m);
                const int cc = first + (phase == 1 ? sh : r < sh ? r : r + 1);
                seq = s0 + l;
                c = __builtin_amdgcn_readlane(cc, l); lo = __builtin_amdgcn_readlane(lo_s, l); hi = __builtin_amdgcn_readlane(hi_s, l);
                return true;
            }
            rest -= __builtin_amdgcn_readlane(incl, 63);
        }
    }
    return false;
}

// Verify: sequence s's first position p0 and the chunks [first, first + n) of C keys that its tokens (consecutive positions)
// meet, up to the one of max_pos. (pos_step: 0 unless each sequence is one row of pos_mode 0.)
__device__ __forceinline__ void seq_chunks(const Problem &p, int C, uint32_t M, int s, int &p0, int &first, int &n) {
    p0 = p.pos_arr ? p.pos_arr[s] : p.base + s * p.pos_step;
    const int p1 = p0 + p.T - 1;
    first = div_by(win_lo(p0, p.window), C, M);
    n = p1 >= 0 ? max(0, min(div_by(p1, C, M), div_by(p.max_pos, C, M)) - first + 1) : 0;
}

// Run number `rest` of at most `slots`: chunk c0 of sequence seq (at position p0, whose chunks end before c_end), and how many chunks the run
// takes from there on, over the following sequences too. The chunks of all sequences, in order, are cut into as many runs as
// there are slots, equal to within one chunk (one chunk each, if they are fewer); or each sequence by itself, where that makes
// no run longer: going on to another sequence costs about 2 us (a window of 1024 keys, 8 sequences x 10 tokens, 256-key chunks:
// 30.2 against 32.2 us). Each chunk starts from a fresh state, so the cut does not show in the results. Cutting each
// sequence by itself in every case left the longest run near the longest sequence's when the sequences were about as many as
// the slots: 48 sequences x 8 tokens of up to 8K keys in 512-key chunks 304 us, now 226.
__device__ __forceinline__ bool find_run(const Problem &p, int C, uint32_t M, int rest, int slots, int &seq, int &p0, int &c0,
                                         int &c_end, int &count) {
    const int lane_ = threadIdx.x & 63;
    int pos = 0, first = 0, n = 0, incl = 0, total = 0;
    for (int s0 = 0; s0 < p.nseq; s0 += 64) {
        n = 0;
        if (s0 + lane_ < p.nseq) seq_chunks(p, C, M, s0 + lane_, pos, first, n);
        incl = wave_scan64(n);
        total += __builtin_amdgcn_readlane(incl, 63);
    }
    if (rest >= min(total, slots)) return false;
    int x = rest;                                           // the run's first chunk, counted over all sequences
    count = 1;
    if (total > slots) {
        const int q = total / slots, r = total - q * slots;
        if (p.nseq <= 64) {
            const int g = r > 0 ? q + 1 : q, k = (n + g - 1) / g, kincl = wave_scan64(k);
            if (__builtin_amdgcn_readlane(kincl, 63) <= slots) {        // each sequence cut by itself
                const unsigned long long hit = __ballot(kincl > rest);
                if (!hit) return false;
                const int l = __builtin_ctzll(hit), j = rest - (kincl - k);
                const int a0 = first + (k > 0 ? j * n / k : 0), a1 = first + (k > 0 ? (j + 1) * n / k : 0);
                seq = l; p0 = __builtin_amdgcn_readlane(pos, l);
                c0 = __builtin_amdgcn_readlane(a0, l); c_end = __builtin_amdgcn_readlane(a1, l);
                count = c_end - c0;
                return true;
            }
        }
        x = rest * q + min(rest, r);
        count = q + (rest < r ? 1 : 0);
    }
    for (int s0 = 0; s0 < p.nseq; s0 += 64) {
        if (p.nseq > 64) {
            n = 0;
            if (s0 + lane_ < p.nseq) seq_chunks(p, C, M, s0 + lane_, pos, first, n);
            incl = wave_scan64(n);
        }
        const unsigned long long hit = __ballot(incl > x);
        if (hit) {
            const int l = __builtin_ctzll(hit), f = __builtin_amdgcn_readlane(first, l), nl = __builtin_amdgcn_readlane(n, l);
            seq = s0 + l; p0 = __builtin_amdgcn_readlane(pos, l);
            c0 = f + x - (__builtin_amdgcn_readlane(incl, l) - nl); c_end = f + nl;
            return true;
        }
        x -= __builtin_amdgcn_readlane(incl, 63);
    }
    return false;
}

// CUs of the current device (0: unknown).
int device_cus();

// Upper bound of the (sequence, chunk) items of a launch: every chunk up to max_pos, or, under a sliding
// window with consecutive token positions, the at most (window + T - 2) / chunk + 2 chunks a window of window + T - 1
// keys meets (a 32K-key cache with a 1K window then launches 6 items per sequence and head, not 128).
inline long long chunk_items_bound(const Problem &p, int chunk) {
    long long per = p.max_pos / chunk + 1;
    if (p.window > 0 && (p.T == 1 || p.pos_mode == 1)) {
        const long long w = ((long long)p.window + p.T - 2) / chunk + 2;
        if (w < per) per = w;
    }
    return per * p.nseq;
}

// Split-KV decode / verify / tree kernels. Verify and tree rows on 16-bit caches at HD <= 256: with slot_runs chunk by
// chunk of each sequence (batch-invariant), otherwise in equal runs over the whole batch (depends on the batch).
hipError_t launch_split(const Problem &p, int chunk, Partials &part, hipStream_t st, bool slot_runs = true);
// Streaming decode kernel (T x GRP <= 16 rows per KV head, HD 128/256, 16-bit cache);
// hipErrorNotSupported for other shapes. Writes chunk partials for launch_combine.
bool decode_stream_supported(const Problem &p);
hipError_t launch_decode_stream(const Problem &p, int chunk, const Partials &part, hipStream_t st);
// The same in fp32 end to end (fp32 Q and cache, fp32 MFMA) for fp32 caches, HD 128/256, T x GRP <= 16.
bool decode_f32_supported(const Problem &p);
hipError_t launch_decode_f32(const Problem &p, int chunk, const Partials &part, hipStream_t st);
// Flash prefill kernel (waves split query rows, K/V tiles shared through LDS). kv_split = 0: one pass per row
// tile writing O directly; kv_split > 0: keys cut at absolute multiples of kv_split, partials + combine.
hipError_t launch_prefill(const Problem &p, int kv_split, const Partials &part, hipStream_t st);
// Verify and tree runs on the prefill tile: up to `chunk` keys per work item, partials for launch_combine (16-bit caches,
// HD 128 / 256, chunk a multiple of 32, consecutive tokens).
bool verify_tile_supported(const Problem &p, int chunk);
hipError_t launch_verify_tile(const Problem &p, int chunk, const Partials &part, hipStream_t st);
// The key split chosen for kv_split = -1 (0: none).
int prefill_auto_split(const Problem &p);
size_t prefill_lds_bytes(int HD);   // dynamic LDS of the HD-wide prefill tile (W = 0)
size_t split_lds_bytes(int HD);     // dynamic LDS of split_kernel at one row block
// LSE combine of split partials for every (row, head).
hipError_t launch_combine(const Problem &p, int chunk, const Partials &part, hipStream_t st);
// Scratch requirement (rows*NQ*ns_cap) of a problem at a given chunk.
size_t partial_rows(const Problem &p, int chunk);

// fp32 scalar kernels of the reference's attention.cuh (small-shape prefill and smem-free decode).
hipError_t launch_scalar_prefill(const float *Q, const float *K, const float *V, float *O, int S, int NQ, int NKV,
                                 int HD, float scale, int window, hipStream_t st);
hipError_t launch_scalar_decode(const float *Q, const float *Kc, const float *Vc, float *O, int nseq, int Sq,
                                int NQ, int NKV, int HD, int base, long kv_stride, const int *base_b, float scale,
                                int window, int reverse, hipStream_t st);
hipError_t launch_scalar_rows(const float *Q, const float *Kc, const float *Vc, float *O, int rows, int NQ, int NKV,
                              int HD, int base, int pos_step, const int *pos_arr, long kv_stride, float scale,
                              int window, int reverse, hipStream_t st);
hipError_t launch_gate_sigmoid(float *y, const float *gate, size_t n, hipStream_t st);
hipError_t launch_kv_store(const float *src, void *dst, size_t n, int kv_dtype, int which, int stats,
                           hipStream_t st);
hipError_t launch_kv_append(const float *ks, const float *vs, void *Kc, void *Vc, int kv_dtype, int nseq, int T,
                            long kv_stride, int row, const int *pos_b, int base, int stats, hipStream_t st);
hipError_t read_kv_stats(unsigned out[4]);
bool norm_rope_shape_ok(int hd, bool rope);
hipError_t launch_norm_rope_store(const float *X, const float *W, void *Y, int y_dtype, int rows, int NH, int hd,
                                  float eps, const float *cosT, const float *sinT, int base, int pos_step,
                                  const int *pos_arr, long slot_stride, long row_stride, bool rope, hipStream_t st);

}  // namespace dgx
