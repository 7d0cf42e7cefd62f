// paged_decode.hip -- split-K paged decode attention on gfx950 MFMA, and the
// reduce kernel that merges the split-K partials.
//
// Math: crates/engine/src/backend/cpu/attention.rs:5-16 (one query row per
// sequence at decode, cpu/mod.rs:314-339).  For query row t, KV head k and
// the G = heads/kv_heads query heads h of k's group:
//   s[j,h] = (K[slot(j),k] . Q[t,kG+h]) * scale          j < row_num_keys[t]
//   out[t,kG+h] = sum_j softmax_j(s[.,h]) V[slot(j),k]
// computed as an online softmax in the exp2 domain (scores pre-multiplied by
// scale*log2 e), fp32 accumulation, bf16 I/O.
//
// Work split.  The keys of each row are cut into splits of `split_keys`
// (a multiple of 32, at most kMaxSplitKeys).  Workgroup (item, k) owns one
// (row, split) for one KV head and all G heads of its group, so every K/V
// byte is read from HBM once: the algorithmic minimum.  An item is one
// 16-byte record (row, split, where the split's block ids start, keys), so
// the workgroup starts its loads after one dependent read.  Its W wavefronts
// take the split's 32-key chunks round robin: chunk c goes to state c % W,
// wavefront c % W's.  A state folds its chunks kSubChunks at a time: each run
// of kSubChunks chunks is an online softmax of its own, and the runs are
// merged in order (fold_state).  Block ids are wave-uniform and
// come from scalar loads.  Each wavefront issues all 16 loads of its next
// chunk before it waits for the current one (two register buffers), so two
// chunks are in flight per wavefront.  The wavefronts merge through LDS at
// the end.  A row with one
// split writes its bf16 output directly; otherwise the workgroup writes an
// fp32 partial (m, l, acc[head_dim]) per head, and decode_reduce_kernel
// merges them:
//   M = max_i m_i,  out = sum_i 2^(m_i-M) acc_i / sum_i 2^(m_i-M) l_i.
//
// Few rows.  A step whose splits are fewer than the CUs runs the longer rows
// one state of a split per workgroup (a "fine" item; W = 4): wavefront s
// takes run s of the state, so that a wavefront walks at most kSubChunks
// chunks in a row and four times the workgroups share the reads; the runs
// are folded through LDS, the partial is the state's, and the merge at the
// end first merges the four states of a split, then the splits.  Operation for
// operation that is what a whole item does, so a row gets the same bits
// either way and batch invariance holds.  Bound: a wavefront's chain of
// chunks (over 1 us each from HBM) and the number of CUs that read at all.
// Two rows of 5000-8100 keys of 8 KV heads of 128 dims are 64 whole items: 25.5 us,
// and 13.9 as 220 fine ones, of a 53 MB read; one row of 8000 keys 27 and
// 13.8 us a call.  Fine items give rows of one split partials too, so only the
// launches that the metadata knows to follow one another run them; any other
// takes the whole items, with the same bits.
//
// The merge.  The last workgroup of a row (and KV head) to finish merges the
// row's partials: they are written and read with
// agent-scope accesses and counted with a relaxed atomic, and no reduce
// launch follows (3 us of GPU time, and 2.5 us of the host's in a small
// call: 13.8 -> 11.1 us for one row of 8000 keys of 64 dims; with shared packs,
// whose workgroups count for each of their rows, in the plans that the host
// chooses it for: merge_packs_in_launch).  (A release and an acquire fence
// per workgroup instead are an L2 writeback and invalidate each time, which
// measured 5-9x slower than the separate launch.)  The counters are the
// upload's, as the plan: zero when it arrives and zero after each launch.
// Packs of one tile, most plans with shared packs, fixed launches, launches
// under capture and launches on another stream than the upload's keep the
// reduce kernel.
// Workgroups are numbered KV head fastest, so the KV heads of one block are
// read at about the same time.
//
// Row packing.  One row's group fills G of the MFMA tile's 16 head columns.
// When the plan finds full splits of several rows over the same physical
// blocks (aliased block-table entries: a shared prefix), one work item
// serves several of them (`pack`; the others are listed in `mates`), and the
// blocks are read once per pack instead of once per row.  Either up to 16 / G
// rows share the tile (column c takes head c % G of row slot c / G), or, in a
// shared pack (shared_split), the workgroup stages each chunk in LDS once and
// each of its 4 wavefronts takes 16 / G rows in its own tile.  MFMA output
// columns and the per-column softmax never mix, and a shared pack keeps the
// register path's per-wavefront states and merge, so every row's result is
// bitwise the one it gets unpacked.
//
// One 32-key chunk (two 16-key blocks b0, b1) of one wavefront:
//   Q.K^T: S^T[key, h] = K[key, :] . Q[h, :] with v_mfma_f32_16x16x32_bf16,
//          A = 16 keys x 32 dims of K (one 16-byte load per lane from the
//          key-major tile), B = Q^T with the G heads in columns 0..G-1 and
//          zeros elsewhere; head_dim/32 MFMAs per 16 keys, two key sets.
//          The A-row -> key assignment is chosen so that lane l ends up
//          holding the scores of head l%16 for keys 8*(l/16) .. +7 of the
//          chunk, in order.
//   softmax: per head, max over the lane's 8 keys and over the 4 lane groups
//          (two xor-shuffles); exp2; the running sum stays per lane and is
//          reduced once at the end.
//   P.V:   O^T[d, h] += V^T[d, key] . P^T[key, h] with 16x16x32 MFMAs:
//          A = 16 dims x 32 keys of V -- lane l reads the 8 keys 8*(l/16)..+7
//          of dim l%16, which are 16 contiguous bytes of the dim-major V tile
//          -- and B = P^T, which is exactly the lane's own 8 probabilities,
//          split into bf16 hi and lo parts (two MFMAs) so P keeps ~16 bits.
//          Output rows are dims, columns heads, so the softmax rescale of the
//          accumulator is lane-local.
// Per chunk and KV head a wavefront moves 16 KiB (hd 128) through 16 global
// loads of 16 bytes per lane and issues 24 MFMAs.
//
// Roofline: HBM.  Algorithmic bytes per row = keys * kv_heads * head_dim * 2 B
// * 2 (K and V) + q and out rows + block-table entries.  The MFMA work is
// <10% of gfx950's bf16 rate even with 12 of 16 head columns padding.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "vo_device.hpp"
#include "vo_kernels.hpp"

namespace vo {
namespace kernels {

namespace {

constexpr int kBS = 16;     // block size of the MFMA path
constexpr int kChunk = 32;  // keys per wavefront iteration
constexpr uint32_t kSubChunks = 4;  // chunks of one run of a state (see fold_state)
// The running max before any key: the lowest finite value, not -inf, so that
// keys scored -inf (weight zero) make no -inf - -inf, wherever they lie; with
// no other key yet, what is summed is zero.
constexpr float kNoMax = -3.40282347e38f;

__device__ __forceinline__ floatx4 mfma16x16x32(bf16x8 a, bf16x8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 load_bf16x8(const uint16_t *p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(p));
}

// K/V tile load.  NT = non-temporal (streaming) loads: on MI355X they raise
// random 4 KiB-tile read bandwidth from ~5.7 to ~6.4 TB/s; used when no KV
// block is read by more than one row of the step, so nothing is lost by not
// keeping the lines in L2.
template <bool NT>
__device__ __forceinline__ bf16x8 load_kv(const uint16_t *p) {
    const u32x4 *v = reinterpret_cast<const u32x4 *>(p);
    if constexpr (NT)
        return __builtin_bit_cast(bf16x8, __builtin_nontemporal_load(v));
    else
        return __builtin_bit_cast(bf16x8, *v);
}

// Max of x over the four lanes l % 16 + 16 g of a column: the row and the
// half-wave swaps of gfx950 hand each lane the other row's (half's) value in
// registers.  (__shfl_xor goes through the LDS permute unit and its latency,
// twice in every chunk's chain.)
__device__ __forceinline__ float column_max(float x) {
    const uint32_t w = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    const float y = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    const uint32_t v = __float_as_uint(y);
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
}

// One chunk's K and V operands, in registers.
template <int HD>
struct Chunk {
    bf16x8 ka[HD / 32];  // first key set (keys 8g + 0..3 land in its result)
    bf16x8 kb[HD / 32];  // second key set (keys 8g + 4..7)
    bf16x8 va[HD / 16];  // V^T rows: dims 16*dt + l%16, keys 8g .. 8g+7
};

// Per-lane element offsets inside one (block, kv head) tile.  K tiles are
// [head_dim/32][16 keys][32 dims] (vo_device.hpp).
struct LaneMap {
    uint32_t k_off;  // Q.K^T A-row m = l%16: key 8*((m>>2)&1) + (m&3), dims 8*(l/16)..
    uint32_t v_off;  // P.V A-row d = l%16: keys 8*(g&1) .. +7 of block g>>1
    bool k_hi;       // A-row m reads block b1 (m >= 8)
    bool v_hi;       // lane group g reads block b1 (g >= 2)
};

template <int HD, bool NT>
__device__ __forceinline__ void load_chunk(Chunk<HD> &r, const uint16_t *k_head,
                                           const uint16_t *v_head, uint64_t block_stride,
                                           uint32_t phys0, uint32_t phys1, const LaneMap &lm) {
    const uint16_t *kp =
        k_head + static_cast<uint64_t>(lm.k_hi ? phys1 : phys0) * block_stride + lm.k_off;
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk) {
        r.ka[kk] = load_kv<NT>(kp + kk * (kBS * 32));
        r.kb[kk] = load_kv<NT>(kp + 4 * 32 + kk * (kBS * 32));
    }
    const uint16_t *vp =
        v_head + static_cast<uint64_t>(lm.v_hi ? phys1 : phys0) * block_stride + lm.v_off;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) r.va[dt] = load_kv<NT>(vp + dt * 16 * kBS);
}

// The step's new key is chunk key kc of r: take its K and V from the new
// rows (nk_row, nv_row: this KV head's head_dim values) instead of the pool,
// which this launch writes them to.  Lane l's K rows are chunk keys
// 16*(m>=8) + 8*((m>>2)&1) + (m&3) (ka) and that + 4 (kb), m = l%16, dims
// 8*(l/16) + 32*kk; its V registers hold keys 8*(l/16) .. +7 of dims
// 16*dt + m (the LaneMap above).
template <int HD>
__device__ __forceinline__ void take_new_key(Chunk<HD> &r, uint32_t kc, const uint16_t *nk_row,
                                             const uint16_t *nv_row, int lane) {
    const uint32_t m = lane & 15;
    const uint32_t g = lane >> 4;
    const uint32_t ka_key = 16 * (m >= 8) + 8 * ((m >> 2) & 1) + (m & 3);
    if (ka_key == kc) {
#pragma unroll
        for (int kk = 0; kk < HD / 32; ++kk)
            r.ka[kk] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(nk_row + 32 * kk + 8 * g));
    }
    if (ka_key + 4 == kc) {
#pragma unroll
        for (int kk = 0; kk < HD / 32; ++kk)
            r.kb[kk] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(nk_row + 32 * kk + 8 * g));
    }
    if ((kc >> 3) == g) {
        const uint32_t i = kc & 7;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) {
            u32x4 w = __builtin_bit_cast(u32x4, r.va[dt]);
            const uint32_t val = nv_row[16 * dt + m];
            const uint32_t sh = 16 * (i & 1);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (q == static_cast<int>(i >> 1)) w[q] = (w[q] & ~(0xffffu << sh)) | (val << sh);
            r.va[dt] = __builtin_bit_cast(bf16x8, w);
        }
    }
}

// One chunk of the online softmax, in two parts: the scores (chunk_qk), then
// the softmax update and P.V (chunk_update).  `nv` = valid keys of this
// lane's group (0..8); the last chunk of a split passes tail = true, with V
// already masked.  Every product and sum is rounded on its own (no fused
// multiply-adds), so that a chunk gets the same bits in every inlined copy:
// the fusion the compiler chooses otherwise depends on the surrounding code
// (whether a product has other uses, as in a tail chunk's masking).
template <int HD>
__device__ __forceinline__ void chunk_qk(const bf16x8 (&ka)[HD / 32], const bf16x8 (&kb)[HD / 32],
                                         const bf16x8 (&qv)[HD / 32], floatx4 &s0, floatx4 &s1) {
    s0 = floatx4{0.f, 0.f, 0.f, 0.f};
    s1 = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk) {
        s0 = mfma16x16x32(ka[kk], qv[kk], s0);
        s1 = mfma16x16x32(kb[kk], qv[kk], s1);
    }
}

// Keys past the end get p = 0; zero their V too, so whatever the pool holds
// there cannot turn 0*x into NaN.
template <int HD>
__device__ __forceinline__ void mask_tail_v(bf16x8 (&va)[HD / 16], int nv) {
    u32x4 mask;
#pragma unroll
    for (int p = 0; p < 4; ++p)
        mask[p] = ((2 * p < nv) ? 0x0000ffffu : 0u) | ((2 * p + 1 < nv) ? 0xffff0000u : 0u);
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt)
        va[dt] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, va[dt]) & mask);
}

// `first` (wave-uniform): the chunk begins a run, whose sums start at zero and
// not at what acc holds.
template <int HD>
__device__ __forceinline__ void chunk_update(const floatx4 &s0, const floatx4 &s1,
                                             const bf16x8 (&va)[HD / 16], bool tail, int nv,
                                             float scale_log2, float &m_run, float &l_run,
                                             floatx4 (&acc)[HD / 16], bool first) {
#pragma clang fp contract(off)
    float sc[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        sc[i] = s0[i];
        sc[4 + i] = s1[i];
    }
    if (tail) {
#pragma unroll
        for (int i = 0; i < 8; ++i) sc[i] = (i < nv) ? sc[i] : -INFINITY;
    }
    float mt = sc[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) mt = fmaxf(mt, sc[i]);
    mt = column_max(mt);
    // at least kNoMax (the scale is positive)
    const float m_new = fmaxf(m_run, mt * scale_log2);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    // P goes to the MFMA as two bf16 parts, hi = bf16(p) and lo = bf16(p - hi),
    // so the probabilities keep ~16 significant bits instead of bf16's 8;
    // bf16 P alone exceeds rtol 1e-2 / atol 2e-3 on rows whose weight sits on
    // a few keys.
    float ps = 0.0f;
    bf16x8 pb_hi, pb_lo;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], scale_log2, -m_new));
        ps += p;
        const __bf16 hi = static_cast<__bf16>(p);
        pb_hi[i] = hi;
        pb_lo[i] = static_cast<__bf16>(p - static_cast<float>(hi));
    }
    l_run = l_run * alpha + ps;
    m_run = m_new;
    if (first) {
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt)
            acc[dt] = mfma16x16x32(va[dt], pb_lo, floatx4{0.f, 0.f, 0.f, 0.f});
    } else {
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) acc[dt] = mfma16x16x32(va[dt], pb_lo, acc[dt] * alpha);
    }
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) acc[dt] = mfma16x16x32(va[dt], pb_hi, acc[dt]);
}

template <int HD>
__device__ __forceinline__ void compute_chunk(Chunk<HD> &r, const bf16x8 (&qv)[HD / 32], bool tail,
                                              int nv, float scale_log2, float &m_run, float &l_run,
                                              floatx4 (&acc)[HD / 16], bool first) {
    floatx4 s0, s1;
    chunk_qk<HD>(r.ka, r.kb, qv, s0, s1);
    if (tail) mask_tail_v<HD>(r.va, nv);
    chunk_update<HD>(s0, s1, r.va, tail, nv, scale_log2, m_run, l_run, acc, first);
}

// (mf, lf, accf) := (mf, lf, accf) merged with the run (m, l, acc) after it.
// Both maxima are at least kNoMax, so neither difference is -inf - -inf.
template <int HD>
__device__ __forceinline__ void fold_state(float &mf, float &lf, floatx4 (&accf)[HD / 16], float m,
                                           float l, const floatx4 (&acc)[HD / 16]) {
#pragma clang fp contract(off)
    const float mx = fmaxf(mf, m);
    const float ef = __builtin_amdgcn_exp2f(mf - mx);
    const float e = __builtin_amdgcn_exp2f(m - mx);
    lf = lf * ef + l * e;
    mf = mx;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j) accf[dt][j] = __builtin_fmaf(accf[dt][j], ef, acc[dt][j] * e);
}

// Split-K partials of a row are merged by the reduce kernel, or by the
// last workgroup of the row's items to finish (`arrivals`; see decode_splitk_kernel).
// In the second form they cross workgroups inside a launch, so they are
// written and read with agent-scope (device-coherent) accesses.
__device__ __forceinline__ void put_f32(float *p, float v, bool agent) {
    if (agent)
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        *p = v;
}

__device__ __forceinline__ void put_f32x4(float *p, floatx4 v, bool agent) {
    if (agent) {
        typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
        const u64x2 w = __builtin_bit_cast(u64x2, v);
        uint64_t *d = reinterpret_cast<uint64_t *>(p);
        __hip_atomic_store(d, static_cast<uint64_t>(w[0]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(d + 1, static_cast<uint64_t>(w[1]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        *reinterpret_cast<floatx4 *>(p) = v;
    }
}

// One state's run in progress (m, l, acc) and the merge of the runs before
// it.  `flush` ends a run, whose successor's first chunk replaces acc; `finish`
// leaves the state in (m, l, acc).  With a wavefront's LDS given to flush and
// finish (room for DT * 64 floatx4), the merged accumulators live there
// between runs, not in registers: 32 registers at head_dim 128, which the two
// chunks in flight need.  They come back in one round of loads, and acc is
// not cleared: with the loads in pairs and 32 clears a flush was longer than a
// chunk's softmax (one row of 900 / 2000 keys of 8 KV heads of 128 dims as
// whole items: 10.8 / 18.6 us, now 10.2 / 17.7; 9.1 / 14.4 without runs at all).
template <int HD>
struct RunState {
    static constexpr int DT = HD / 16;
    float m, l, mf, lf;
    floatx4 acc[DT], accf[DT];

    __device__ __forceinline__ void reset() {
        m = kNoMax;
        l = 0.0f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    // In registers; `first`: nothing in accf yet.
    __device__ __forceinline__ void flush(bool first) {
        if (first) {
            mf = m;
            lf = l;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) accf[dt] = acc[dt];
        } else {
            fold_state<HD>(mf, lf, accf, m, l, acc);
        }
        m = kNoMax;
        l = 0.0f;
    }
    __device__ __forceinline__ void finish(bool first) {
        if (first) return;
        fold_state<HD>(mf, lf, accf, m, l, acc);
        m = mf;
        l = lf;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = accf[dt];
    }
    // The same with accf in lds[dt * 64 + lane]; `first`: nothing there yet.
    __device__ __forceinline__ void flush(floatx4 *lds, int lane, bool first) {
        finish(lds, lane, first);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) lds[dt * 64 + lane] = acc[dt];
        mf = m;
        lf = l;
        m = kNoMax;
        l = 0.0f;
    }
    __device__ __forceinline__ void finish(const floatx4 *lds, int lane, bool first) {
        if (first) return;
        floatx4 f[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) f[dt] = lds[dt * 64 + lane];
        __builtin_amdgcn_sched_barrier(0);  // all loads, then one wait
        fold_state<HD>(mf, lf, f, m, l, acc);
        m = mf;
        l = lf;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = f[dt];
    }
};

// Keeps the scheduler from moving instructions across this point: the next
// chunk's loads are all issued before the current chunk's first wait.
__device__ __forceinline__ void issue_fence() { __builtin_amdgcn_sched_barrier(0); }

// A shared pack: one full split whose blocks the rows of a pack all read
// (an aliased prefix), for up to W * (16 / G) rows.  Each wavefront owns one
// 16-column tile (rows w * 16/G ..) and walks every chunk of the split, so
// the workgroup reads each K/V byte once for all of its rows instead of once
// per wavefront.  A chunk (two blocks: K b0, K b1, V b0, V b1, one tile
// each) is copied into LDS by LDS DMA, 16 bytes per lane from the lane's own
// global address, through a ring of four stages; the workgroup takes one
// chunk per barrier while the next three load.  The wavefronts then read their operands from LDS at
// the positions the register path loads from the pool and run its
// compute_chunk.  The chunks of state 0 (c % W == 0) come first, then those
// of state 1 and so on, each in the register path's runs, and the W states
// are merged as that path merges its wavefronts, so every column's result is
// the register path's, bit for bit.
//
// LDS bank spread: within a tile, 16-byte unit x sits at unit swz(x).  K
// unit x = 64 kk + 4 key + j (dims 8 j.. of 32-dim chunk kk): j ^= 2 (key >>
// 3) ^ (block & 1), so the 16 lanes of one read phase (keys 0-3 and 8-11 of
// two blocks) fill 16 distinct 4-bank groups.  V unit x = 2 dim + half:
// half ^= (dim >> 3) & 1.  Both are involutions on the low bits, so the DMA
// reads global unit swz(u) into LDS unit u.
// Floats per column of the wavefronts' merge buffer: 4 more than head_dim, so
// that the 16 columns of one store phase fall into 16 different bank groups.
template <int HD>
constexpr uint32_t kAccStride = HD + 4;

// A shared pack keeps W softmax states per wavefront (W x 32 registers at
// head_dim 128), and its four stages also hold the register path's merge:
// exactly 4 wavefronts (with 2 the four-stage loop no longer fits two
// wavefronts per SIMD).
constexpr int kSharedWaves = 4;

template <int HD>
struct SharedStage {
    static constexpr uint32_t TB = kBS * HD * 2;   // bytes of one (block, KV head) tile
    static constexpr uint32_t BYTES = 4 * TB;      // K b0, K b1, V b0, V b1
    __device__ static __forceinline__ uint32_t swz_k(uint32_t x, uint32_t b) {
        return x ^ (((x >> 5) & 1u) << 1) ^ (b & 1u);
    }
    __device__ static __forceinline__ uint32_t swz_v(uint32_t x) { return x ^ ((x >> 4) & 1u); }
};

template <int HD, int W>
__device__ __forceinline__ void shared_split(
    const uint16_t *__restrict__ k_pool, const uint16_t *__restrict__ v_pool, uint32_t kv_heads,
    uint32_t kvh, uint32_t item, const u32x4 rec, const uint32_t *__restrict__ tables,
    const uint32_t *__restrict__ row_info, uint32_t split_keys, const uint16_t *__restrict__ q,
    uint16_t *__restrict__ out, float *__restrict__ part_acc, float *__restrict__ part_ml,
    uint32_t num_heads, uint32_t group, float scale_log2, const uint32_t *__restrict__ mates,
    uint32_t pack, uint8_t *__restrict__ st0, uint8_t *__restrict__ st1,
    uint8_t *__restrict__ st2, uint8_t *__restrict__ st3, bool agent) {
#pragma clang fp contract(off)  // the merge below rounds as the register path's does
    constexpr int KK = HD / 32;
    constexpr int DT = HD / 16;
    using S = SharedStage<HD>;
    constexpr uint32_t kTile = kBS * HD;
    constexpr int NI = S::BYTES / 1024 / W;  // DMA instructions per wavefront and chunk
    static_assert(S::BYTES % (1024 * W) == 0 && NI <= 15, "chunk DMA split");
    constexpr uint32_t KIB_PER_TILE = S::TB / 1024;

    const uint32_t row = uniform_u32(rec[0]);
    const uint32_t split = uniform_u32(rec[1]);  // a pack is never a fine item
    const uint32_t *table = tables + uniform_u32(rec[2]);
    const uint32_t nchunks = split_keys / kChunk;  // a full split
    // The split's block ids (at most kMaxSplitKeys / 16 = 256), 64 per
    // register across the lanes, read before the first DMA; a chunk's two ids
    // are then v_readlane'd.  (Loads from the table after an LDS DMA would be
    // vector loads, and every wait for one would also wait for the DMA.)
    constexpr int TV = kMaxSplitKeys / kBS / 64;
    const uint32_t nblk = 2 * nchunks;
    uint32_t tv[TV];
#pragma unroll
    for (int k = 0; k < TV; ++k) {
        const uint32_t i = 64 * k + static_cast<uint32_t>(threadIdx.x & 63);
        tv[k] = i < nblk ? table[i] : 0u;
    }
    auto block_id = [&](uint32_t i) {  // i < nblk, wave-uniform
        uint32_t b = __builtin_amdgcn_readlane(tv[0], i & 63);
#pragma unroll
        for (int k = 1; k < TV; ++k) {
            const uint32_t bk = __builtin_amdgcn_readlane(tv[k], i & 63);
            b = (i >> 6) == static_cast<uint32_t>(k) ? bk : b;
        }
        return b;
    };
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane & 15;
    const int g = lane >> 4;

    // This wavefront's columns: row slot wave * R + h / G, head h % G, with
    // R = ceil(pack / W) <= 16 / G rows per wavefront.
    const uint32_t per_wave = (pack + W - 1) / W;
    const uint32_t hslot = static_cast<uint32_t>(h) / group;
    const uint32_t pslot = static_cast<uint32_t>(wave) * per_wave + hslot;
    const uint32_t hh = static_cast<uint32_t>(h) - hslot * group;
    uint32_t crow = kNoMate;
    if (hslot < per_wave) {
        if (pslot == 0)
            crow = row;
        else if (pslot < pack)
            crow = mates[(pack - 1) * item + pslot - 1];
    }
    const bool head_ok = crow != kNoMate;
    // Whether any column of this wavefront is live (wave-uniform).
    const bool wave_live = __builtin_amdgcn_ballot_w64(head_ok) != 0;
    const uint32_t qhead = kvh * group + hh;
    bf16x8 qv[KK];
    {
        const uint16_t *qp = q + (static_cast<uint64_t>(head_ok ? crow : row) * num_heads + qhead) * HD + 8 * g;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) qv[kk] = head_ok ? load_bf16x8(qp + 32 * kk) : bf16x8{};
    }
    u32x2 cinfo = {0u, 0u};
    if (head_ok) cinfo = *reinterpret_cast<const u32x2 *>(row_info + 2 * static_cast<uint64_t>(crow));

    // DMA: instruction i of wavefront w copies KiB qi = i * W + w of the
    // stage: tile qi / KIB_PER_TILE (K b0, K b1, V b0, V b1), its KiB qi %
    // KIB_PER_TILE; lane unit u of that tile reads global unit swz(u).
    uint32_t dma_off[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const uint32_t qi = static_cast<uint32_t>(i * W + wave);
        const uint32_t t = qi / KIB_PER_TILE;
        const uint32_t u = (qi % KIB_PER_TILE) * 64 + lane;
        dma_off[i] = 16 * (t < 2 ? S::swz_k(u, t) : S::swz_v(u));
    }
    const uint64_t block_stride = static_cast<uint64_t>(kv_heads) * kTile;
    auto dma_chunk = [&](uint8_t *stage, uint32_t c) {
        const uint32_t b0 = block_id(2 * c);
        const uint32_t b1 = block_id(2 * c + 1);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const uint32_t qi = static_cast<uint32_t>(i * W + wave);
            const uint32_t t = qi / KIB_PER_TILE;
            const uint16_t *pool = t < 2 ? k_pool : v_pool;
            const uint32_t blk = (t & 1) ? b1 : b0;
            dma16(pool + static_cast<uint64_t>(blk) * block_stride + static_cast<uint64_t>(kvh) * kTile,
                  S::TB, stage + qi * 1024, dma_off[i]);
        }
    };

    // LDS read offsets of this lane (the register path's LaneMap positions,
    // swizzled): K A-row m = l % 16 reads key 8((m >> 2) & 1) + (m & 3) of
    // block m >= 8, dims 8 g .. of chunk kk (+64 kk units) and the key + 4
    // (+16 units); V lane reads dim 16 dt + m (+32 dt units), keys 8 (g & 1)
    // .. +7 of block g >= 2.
    const uint32_t m = static_cast<uint32_t>(h);
    const uint32_t kb_hi = m >= 8 ? 1u : 0u;
    const uint32_t kx = (8 * ((m >> 2) & 1) + (m & 3)) * 4 + static_cast<uint32_t>(g);
    const uint32_t k_rd = kb_hi * S::TB + 16 * S::swz_k(kx, kb_hi);
    const uint32_t vb_hi = g >= 2 ? 1u : 0u;
    const uint32_t vx = 2 * m + static_cast<uint32_t>(g & 1);
    const uint32_t v_rd = (2 + vb_hi) * S::TB + 16 * S::swz_v(vx);

    // State w: the (m, l, acc) the register path's wavefront w keeps, in the
    // same order, merged at the end as that path merges its wavefronts.  So a
    // row's bits do not depend on whether it was packed.
    float ms[W], ls[W];
    floatx4 as[W][DT];

    auto read_k = [&](const uint8_t *cur, bf16x8 (&ka)[KK], bf16x8 (&kb)[KK])
        __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            ka[kk] = *reinterpret_cast<const bf16x8 *>(cur + k_rd + 1024 * kk);
            kb[kk] = *reinterpret_cast<const bf16x8 *>(cur + k_rd + 1024 * kk + 256);
        }
    };
    auto read_v = [&](const uint8_t *cur, bf16x8 (&va)[DT]) __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) va[dt] = *reinterpret_cast<const bf16x8 *>(cur + v_rd + 512 * dt);
    };
    // Step t stages chunk chunk_of(t): `per` steps for each state, padded to
    // the four stages (steps without a chunk stage the last one and compute
    // nothing).
    const uint32_t per = (nchunks + 4 * W - 1) / (4 * W) * 4;
    auto chunk_of = [&](uint32_t t) { return (t % per) * W + t / per; };
    auto staged = [&](uint32_t t) { return min(chunk_of(min(t, W * per - 1)), nchunks - 1); };
    static_assert(W == 4, "four stages");
    dma_chunk(st0, staged(0));
    dma_chunk(st1, staged(1));
    dma_chunk(st2, staged(2));
    auto state = [&](auto w_c) __attribute__((always_inline)) {
        constexpr int w = decltype(w_c)::value;
        RunState<HD> rs;
        rs.reset();
        // One chunk per step: step t waits for its chunk (the DMA of the next
        // two may fly on) and for every wavefront to be done with the step
        // before, refills that stage with the chunk three steps on and
        // computes.  Every step issues its DMA, so the wait count stays
        // uniform.
        auto one = [&](auto s_c, uint32_t k) __attribute__((always_inline)) {
            constexpr int sidx = decltype(s_c)::value;
            uint8_t *__restrict__ cur = sidx == 0 ? st0 : sidx == 1 ? st1 : sidx == 2 ? st2 : st3;
            uint8_t *__restrict__ nxt = sidx == 0 ? st3 : sidx == 1 ? st0 : sidx == 2 ? st1 : st2;
            wait_barrier<2 * NI>();
            dma_chunk(nxt, staged(w * per + k + 3));
            if (!wave_live || k * W + w >= nchunks) return;
            if (sidx == 0 && k != 0) rs.flush(k == kSubChunks);  // runs of kSubChunks == 4 chunks
            bf16x8 ka[KK], kb[KK], va[DT];
            floatx4 sa0, sa1;
            read_k(cur, ka, kb);
            chunk_qk<HD>(ka, kb, qv, sa0, sa1);
            read_v(cur, va);
            chunk_update<HD>(sa0, sa1, va, false, 8, scale_log2, rs.m, rs.l, rs.acc, sidx == 0);
        };
        static_assert(kSubChunks == 4, "a run is one turn of the stages");
        for (uint32_t k = 0; k < per; k += 4) {
            one(std::integral_constant<int, 0>{}, k);
            one(std::integral_constant<int, 1>{}, k + 1);
            one(std::integral_constant<int, 2>{}, k + 2);
            one(std::integral_constant<int, 3>{}, k + 3);
        }
        if (wave_live) rs.finish(nchunks <= W * kSubChunks + w);  // at most one run
        ms[w] = rs.m;
        ls[w] = rs.l;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) as[w][dt] = rs.acc[dt];
    };
    state(std::integral_constant<int, 0>{});
    state(std::integral_constant<int, 1>{});
    state(std::integral_constant<int, 2>{});
    state(std::integral_constant<int, 3>{});
    // The DMA past the last chunk must land before the workgroup's LDS is
    // released.
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));

    if (!head_ok) return;
    // The register path's merge of its W wavefronts, per element.
#pragma unroll
    for (int w = 0; w < W; ++w) {
        ls[w] += __shfl_xor(ls[w], 16, 64);
        ls[w] += __shfl_xor(ls[w], 32, 64);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; ++w) mx = fmaxf(mx, ms[w]);
    float den = 0.0f;
    floatx4 num[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) num[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const float e = __builtin_amdgcn_exp2f(ms[w] - mx);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int j = 0; j < 4; ++j) num[dt][j] += e * as[w][dt][j];
        den += e * ls[w];
    }
    if (cinfo[1] == 1) {
        uint16_t *op = out + static_cast<uint64_t>(crow) * num_heads * HD +
                       static_cast<uint64_t>(qhead) * HD + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int j = 0; j < 4; ++j) op[16 * dt + j] = f32_to_bf16_bits(num[dt][j] / den);
    } else {
        const uint64_t part = static_cast<uint64_t>(cinfo[0] + split) * num_heads + qhead;
        float *ap = part_acc + part * HD + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) put_f32x4(ap + 16 * dt, num[dt], agent);
        if (g == 0) {
            put_f32(part_ml + 2 * part, mx, agent);
            put_f32(part_ml + 2 * part + 1, den, agent);
        }
    }
}

// A shared pack in wavefront pairs.  The same staged chunks and the same
// four softmax states as shared_split, but each 16-column tile has two
// wavefronts: the one of parity 0 keeps states 0 and 2 (chunks 4k and
// 4k + 2), the one of parity 1 states 1 and 3 (chunks 4k + 1, 4k + 3).  One
// step stages two chunks and each
// wavefront of a pair computes one of them, so a wavefront walks half of the
// split's chunks: first the chunks of states 0 and 1 (4k, 4k + 1), then those of states
// 2 and 3, so that a wavefront has one run in progress.  The workgroup holds W / 2 tiles, so a pack has W / 2 *
// (16 / G) rows.  Every state still takes its chunks in increasing order,
// and the four states are merged in the order 0..3 with the register path's
// arithmetic, so a row's bits are the register path's, as in shared_split.
// Two chunks are consumed per step, so the DMA of a step's pair is issued
// one step ahead (the four stages hold two pairs).
template <int HD, int W>
__device__ __forceinline__ void shared_split_pairs(
    const uint16_t *__restrict__ k_pool, const uint16_t *__restrict__ v_pool, uint32_t kv_heads,
    uint32_t kvh, uint32_t item, const u32x4 rec, const uint32_t *__restrict__ tables,
    const uint32_t *__restrict__ row_info, uint32_t split_keys, const uint16_t *__restrict__ q,
    uint16_t *__restrict__ out, float *__restrict__ part_acc, float *__restrict__ part_ml,
    uint32_t num_heads, uint32_t group, float scale_log2, const uint32_t *__restrict__ mates,
    uint32_t pack, uint8_t *__restrict__ st0, uint8_t *__restrict__ st1,
    uint8_t *__restrict__ st2, uint8_t *__restrict__ st3, bool agent) {
#pragma clang fp contract(off)  // the merge below rounds as the register path's does
    constexpr int KK = HD / 32;
    constexpr int DT = HD / 16;
    using S = SharedStage<HD>;
    constexpr uint32_t kTile = kBS * HD;
    constexpr int NI = S::BYTES / 1024 / W;  // DMA instructions per wavefront and chunk
    static_assert(W == 4 && S::BYTES % (1024 * W) == 0 && 2 * NI <= 15, "chunk DMA split");
    constexpr uint32_t KIB_PER_TILE = S::TB / 1024;
    constexpr uint32_t kTiles = W / 2;
    // The partner's two states go through the stages: per tile, DT x 64
    // lanes of floatx4 per state (one stage), and (m, l) per state and lane.
    static_assert(2 * DT * 64 * 16 <= S::BYTES && kTiles * 4 * 64 * 4 <= S::BYTES,
                  "pair exchange fits the stages");
    // The packs set the launch's length and share each CU with a
    // register-path workgroup that has slack: their wavefronts win the
    // SIMDs' issue arbitration.
    __builtin_amdgcn_s_setprio(3);

    const uint32_t row = uniform_u32(rec[0]);
    const uint32_t split = uniform_u32(rec[1]);  // a pack is never a fine item
    const uint32_t *table = tables + uniform_u32(rec[2]);
    const uint32_t nchunks = split_keys / kChunk;  // a full split
    constexpr int TV = kMaxSplitKeys / kBS / 64;
    const uint32_t nblk = 2 * nchunks;
    uint32_t tv[TV];
#pragma unroll
    for (int k = 0; k < TV; ++k) {
        const uint32_t i = 64 * k + static_cast<uint32_t>(threadIdx.x & 63);
        tv[k] = i < nblk ? table[i] : 0u;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane & 15;
    const int g = lane >> 4;
    const uint32_t tile = static_cast<uint32_t>(wave) >> 1;
    const uint32_t par = static_cast<uint32_t>(wave) & 1;

    // This tile's columns: row slot tile * R + h / G, head h % G, with
    // R = ceil(pack / tiles) <= 16 / G rows per tile.
    const uint32_t per_tile = (pack + kTiles - 1) / kTiles;
    const uint32_t hslot = static_cast<uint32_t>(h) / group;
    const uint32_t pslot = tile * per_tile + hslot;
    const uint32_t hh = static_cast<uint32_t>(h) - hslot * group;
    uint32_t crow = kNoMate;
    if (hslot < per_tile) {
        if (pslot == 0)
            crow = row;
        else if (pslot < pack)
            crow = mates[(pack - 1) * item + pslot - 1];
    }
    const bool head_ok = crow != kNoMate;
    const bool wave_live = __builtin_amdgcn_ballot_w64(head_ok) != 0;
    const uint32_t qhead = kvh * group + hh;
    bf16x8 qv[KK];
    {
        const uint16_t *qp = q + (static_cast<uint64_t>(head_ok ? crow : row) * num_heads + qhead) * HD + 8 * g;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) qv[kk] = head_ok ? load_bf16x8(qp + 32 * kk) : bf16x8{};
    }
    u32x2 cinfo = {0u, 0u};
    if (head_ok) cinfo = *reinterpret_cast<const u32x2 *>(row_info + 2 * static_cast<uint64_t>(crow));

    // DMA as in shared_split: instruction i of wavefront w copies KiB i * W
    // + w of a chunk's stage.
    uint32_t dma_off[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const uint32_t qi = static_cast<uint32_t>(i * W + wave);
        const uint32_t t = qi / KIB_PER_TILE;
        const uint32_t u = (qi % KIB_PER_TILE) * 64 + lane;
        dma_off[i] = 16 * (t < 2 ? S::swz_k(u, t) : S::swz_v(u));
    }
    const uint64_t block_stride = static_cast<uint64_t>(kv_heads) * kTile;
    auto block_id = [&](uint32_t i) {  // i < nblk, wave-uniform
        uint32_t b = __builtin_amdgcn_readlane(tv[0], i & 63);
#pragma unroll
        for (int k = 1; k < TV; ++k) {
            const uint32_t bk = __builtin_amdgcn_readlane(tv[k], i & 63);
            b = (i >> 6) == static_cast<uint32_t>(k) ? bk : b;
        }
        return b;
    };
    auto dma_chunk = [&](uint8_t *stage, uint32_t c) __attribute__((always_inline)) {
        const uint32_t b0 = block_id(2 * c);
        const uint32_t b1 = block_id(2 * c + 1);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const uint32_t qi = static_cast<uint32_t>(i * W + wave);
            const uint32_t t = qi / KIB_PER_TILE;
            const uint16_t *pool = t < 2 ? k_pool : v_pool;
            const uint32_t blk = (t & 1) ? b1 : b0;
            dma16(pool + static_cast<uint64_t>(blk) * block_stride + static_cast<uint64_t>(kvh) * kTile,
                  S::TB, stage + qi * 1024, dma_off[i]);
        }
    };

    // LDS read offsets: shared_split's.
    const uint32_t m = static_cast<uint32_t>(h);
    const uint32_t kb_hi = m >= 8 ? 1u : 0u;
    const uint32_t kx = (8 * ((m >> 2) & 1) + (m & 3)) * 4 + static_cast<uint32_t>(g);
    const uint32_t k_rd = kb_hi * S::TB + 16 * S::swz_k(kx, kb_hi);
    const uint32_t vb_hi = g >= 2 ? 1u : 0u;
    const uint32_t vx = 2 * m + static_cast<uint32_t>(g & 1);
    const uint32_t v_rd = (2 + vb_hi) * S::TB + 16 * S::swz_v(vx);

    // Local state i is state par + 2 i.
    float ms[2], ls[2];
    floatx4 as[2][DT];
    auto compute = [&](auto first_c, const uint8_t *cur, RunState<HD> &rs)
        __attribute__((always_inline)) {
        constexpr bool first = decltype(first_c)::value;  // of a run
        bf16x8 ka[KK], kb[KK], va[DT];
        floatx4 sa0, sa1;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            ka[kk] = *reinterpret_cast<const bf16x8 *>(cur + k_rd + 1024 * kk);
            kb[kk] = *reinterpret_cast<const bf16x8 *>(cur + k_rd + 1024 * kk + 256);
        }
        chunk_qk<HD>(ka, kb, qv, sa0, sa1);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) va[dt] = *reinterpret_cast<const bf16x8 *>(cur + v_rd + 512 * dt);
        chunk_update<HD>(sa0, sa1, va, false, 8, scale_log2, rs.m, rs.l, rs.acc, first);
    };
    // Step t stages chunks pair_of(t) and the next: `per` steps (whole runs)
    // for the states 0 and 1, then as many for 2
    // and 3; a step past a state's last chunk stages the split's last one and
    // computes nothing.
    const uint32_t per = (nchunks + 4 * kSubChunks - 1) / (4 * kSubChunks) * kSubChunks;
    auto pair_of = [&](uint32_t t) { return t < per ? 4 * t : 4 * (t - per) + 2; };
    // Step t: wait for its two chunks (the only DMA in flight), then
    // for every wavefront to be done with the step before, refill that
    // step's stages with the next step's chunks, and compute chunk pair_of(t)
    // + par.  Each stage is named in its
    // own branch, so that the compiler tells the stage being read from the
    // ones the DMA fills.  Every step issues its DMA (past the last step
    // the chunks are the split's last).
    // The two phases run in a rolled loop, a run to a turn: the code of a
    // chunk is large, and the instruction cache is shared with the register
    // path's workgroups.
    dma_chunk(st0, 0);
    dma_chunk(st1, min(1u, nchunks - 1));
#pragma unroll 1
    for (uint32_t i = 0; i < 2; ++i) {
        RunState<HD> rs;
        rs.reset();
        auto step = [&](auto s_run, uint32_t k) __attribute__((always_inline)) {
            constexpr int in_run = decltype(s_run)::value;  // k % kSubChunks
            constexpr int sp = in_run % 2;
            using First = std::integral_constant<bool, in_run == 0>;
            const uint32_t nx = pair_of(min(i * per + k + 1, 2 * per - 1));
            wait_barrier<0>();
            dma_chunk(sp ? st0 : st2, min(nx, nchunks - 1));
            dma_chunk(sp ? st1 : st3, min(nx + 1, nchunks - 1));
            if (!wave_live || 4 * k + 2 * i + par >= nchunks) return;
            if (in_run == 0 && k != 0) rs.flush(k == kSubChunks);
            if (par == 0)
                compute(First{}, sp ? st2 : st0, rs);
            else
                compute(First{}, sp ? st3 : st1, rs);
        };
        static_assert(kSubChunks == 4, "a run's steps");
#pragma unroll 1
        for (uint32_t k = 0; k < per; k += 4) {
            step(std::integral_constant<int, 0>{}, k);
            step(std::integral_constant<int, 1>{}, k + 1);
            step(std::integral_constant<int, 2>{}, k + 2);
            step(std::integral_constant<int, 3>{}, k + 3);
        }
        if (wave_live) rs.finish(nchunks <= 4 * kSubChunks + 2 * i + par);  // at most one run
        if (i == 0) {
            ms[0] = rs.m;
            ls[0] = rs.l;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) as[0][dt] = rs.acc[dt];
        } else {
            ms[1] = rs.m;
            ls[1] = rs.l;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) as[1][dt] = rs.acc[dt];
        }
    }
    // The DMA past the last chunk must land before the stages are reused.
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));
    // The running sums are per lane group (the four lanes of a column are
    // all live or all not).
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        ls[i] += __shfl_xor(ls[i], 16, 64);
        ls[i] += __shfl_xor(ls[i], 32, 64);
    }
    // The parity-1 wavefront hands its states to its partner through the
    // stages, once every wavefront is done reading them.
    __syncthreads();
    floatx4 *xa = reinterpret_cast<floatx4 *>(tile == 0 ? st0 : st1);  // [2][DT][64]
    float *xml = reinterpret_cast<float *>(st2) + tile * 4 * 64;     // [2][m, l][64]
    if (par == 1 && head_ok) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) xa[(i * DT + dt) * 64 + lane] = as[i][dt];
            xml[(2 * i) * 64 + lane] = ms[i];
            xml[(2 * i + 1) * 64 + lane] = ls[i];
        }
    }
    __syncthreads();
    if (par == 1 || !head_ok) return;

    // The register path's merge of its W = 4 wavefronts' states, in order
    // 0..3: state 2i is this wavefront's local state i, state 2i + 1 the
    // partner's.
    float sm[4], sl[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        sm[2 * i] = ms[i];
        sl[2 * i] = ls[i];
        sm[2 * i + 1] = xml[(2 * i) * 64 + lane];
        sl[2 * i + 1] = xml[(2 * i + 1) * 64 + lane];
    }
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) mx = fmaxf(mx, sm[w]);
    float den = 0.0f;
    floatx4 num[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) num[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const float e = __builtin_amdgcn_exp2f(sm[w] - mx);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const floatx4 a = (w & 1) ? xa[((w >> 1) * DT + dt) * 64 + lane] : as[w >> 1][dt];
#pragma unroll
            for (int j = 0; j < 4; ++j) num[dt][j] += e * a[j];
        }
        den += e * sl[w];
    }
    if (cinfo[1] == 1) {
        uint16_t *op = out + static_cast<uint64_t>(crow) * num_heads * HD +
                       static_cast<uint64_t>(qhead) * HD + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int j = 0; j < 4; ++j) op[16 * dt + j] = f32_to_bf16_bits(num[dt][j] / den);
    } else {
        const uint64_t part = static_cast<uint64_t>(cinfo[0] + split) * num_heads + qhead;
        float *ap = part_acc + part * HD + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) put_f32x4(ap + 16 * dt, num[dt], agent);
        if (g == 0) {
            put_f32(part_ml + 2 * part, mx, agent);
            put_f32(part_ml + 2 * part + 1, den, agent);
        }
    }
}

template <bool AGENT>
__device__ __forceinline__ float get_f32(const float *p) {
    if constexpr (AGENT)
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        return *p;
}

template <bool AGENT>
__device__ __forceinline__ floatx4 get_f32x4(const float *p) {
    if constexpr (AGENT) {
        typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
        const uint64_t *d = reinterpret_cast<const uint64_t *>(p);
        u64x2 w;
        w[0] = __hip_atomic_load(d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        w[1] = __hip_atomic_load(d + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return __builtin_bit_cast(floatx4, w);
    } else {
        return *reinterpret_cast<const floatx4 *>(p);
    }
}

// States of a split of `keys` keys that hold keys: the fine items it has.
__device__ __forceinline__ uint32_t split_states(uint32_t keys) {
    return min((keys + kChunk - 1) / kChunk, static_cast<uint32_t>(kSharedWaves));
}

// Merges one row's partials for dims d .. d + 3 of query head qh and writes
// them.  The splits are folded in order with a running max; a fine row's
// split is first the merge of its states, as the split kernel merges its
// wavefronts, so the result depends on the row's keys only.  Four partials
// of a row of up to four splits, and eight of another or of a fine row, are
// loaded before the first is used.
template <int HD, bool AGENT>
__device__ __forceinline__ void merge_row(const float *part_acc, const float *part_ml,
                                          uint32_t first, uint32_t nsplit, bool fine, uint32_t nk,
                                          uint32_t split_keys, uint32_t num_heads, uint32_t qh,
                                          uint32_t d, uint16_t *out) {
#pragma clang fp contract(off)
    constexpr int W = kSharedWaves;
    constexpr int U = 8;
    float mx = -INFINITY, den = 0.0f;
    floatx4 num = {0.f, 0.f, 0.f, 0.f};
    float m[U], l[U];
    floatx4 a[U];
    auto load = [&](int u, uint32_t slot) {
        const uint64_t part = static_cast<uint64_t>(slot) * num_heads + qh;
        m[u] = get_f32<AGENT>(part_ml + 2 * part);
        l[u] = get_f32<AGENT>(part_ml + 2 * part + 1);
        a[u] = get_f32x4<AGENT>(part_acc + part * HD + d);
    };
    auto fold = [&](float mi, float li, const floatx4 &ai) {
        const float m_new = fmaxf(mx, mi);
        const float scale_old = __builtin_amdgcn_exp2f(mx - m_new);
        const float e = __builtin_amdgcn_exp2f(mi - m_new);
        den = den * scale_old + e * li;
        num = num * scale_old + ai * e;
        mx = m_new;
    };
    if (!fine) {
        auto rounds = [&](auto r_c) __attribute__((always_inline)) {
            constexpr uint32_t R = decltype(r_c)::value;  // splits per round
            for (uint32_t i = 0; i < nsplit; i += R) {
#pragma unroll
                for (uint32_t u = 0; u < R; ++u) load(u, first + min(i + u, nsplit - 1));
#pragma unroll
                for (uint32_t u = 0; u < R; ++u)
                    if (i + u < nsplit) fold(m[u], l[u], a[u]);
            }
        };
        if (nsplit <= 4)
            rounds(std::integral_constant<uint32_t, 4>{});
        else
            rounds(std::integral_constant<uint32_t, U>{});
    } else {
        constexpr int S = U / W;  // splits per round
        for (uint32_t i = 0; i < nsplit; i += S) {
            uint32_t states[S];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const uint32_t sp = min(i + s, nsplit - 1);
                states[s] = split_states(min(nk - sp * split_keys, split_keys));
                // Past the split's states: its first one, not used.
#pragma unroll
                for (int w = 0; w < W; ++w)
                    load(s * W + w, first + W * sp + (static_cast<uint32_t>(w) < states[s] ? w : 0));
            }
#pragma unroll
            for (int s = 0; s < S; ++s) {
                if (i + s >= nsplit) break;
                float ms = -INFINITY;
#pragma unroll
                for (int w = 0; w < W; ++w)
                    if (static_cast<uint32_t>(w) < states[s]) ms = fmaxf(ms, m[s * W + w]);
                float ds = 0.0f;
                floatx4 ns = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    if (static_cast<uint32_t>(w) < states[s]) {
                        const float e = __builtin_amdgcn_exp2f(m[s * W + w] - ms);
#pragma unroll
                        for (int j = 0; j < 4; ++j) ns[j] += e * a[s * W + w][j];
                        ds += e * l[s * W + w];
                    }
                }
                if (nsplit == 1) {  // as the split kernel's own output
                    num = ns;
                    den = ds;
                } else {
                    fold(ms, ds, ns);
                }
            }
        }
    }
    u32x2 packed;
    if (fine && nsplit == 1) {
        packed[0] = f32_to_bf16_bits(num[0] / den) |
                    (static_cast<uint32_t>(f32_to_bf16_bits(num[1] / den)) << 16);
        packed[1] = f32_to_bf16_bits(num[2] / den) |
                    (static_cast<uint32_t>(f32_to_bf16_bits(num[3] / den)) << 16);
    } else {
        const float inv = 1.0f / den;
        packed[0] = f32_to_bf16_bits(num[0] * inv) |
                    (static_cast<uint32_t>(f32_to_bf16_bits(num[1] * inv)) << 16);
        packed[1] = f32_to_bf16_bits(num[2] * inv) |
                    (static_cast<uint32_t>(f32_to_bf16_bits(num[3] * inv)) << 16);
    }
    *reinterpret_cast<u32x2 *>(out + d) = packed;
}

// The kernels of a launch: one without packs (single rows, fine items)
// and one for each form of shared packs beside single rows,
// so that neither carries the other's code, which would not fit half the
// instruction cache (22 and 33 KB at head_dim 128; all in one 50 KB, and the
// 64-row decode step 0.9% longer).
enum PackKind : int { kNoPacks = 0, kPairPacks = 1, kSinglePacks = 2 };

template <int HD, int W, bool NT, int PACKS>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2))) void
decode_splitk_kernel(const uint16_t *__restrict__ k_pool, const uint16_t *__restrict__ v_pool,
                     uint32_t kv_heads, const uint32_t *__restrict__ tables,
                     const uint32_t *__restrict__ work,
                     const uint32_t *__restrict__ row_info, uint32_t split_keys,
                     const uint16_t *__restrict__ q, uint16_t *__restrict__ out,
                     float *__restrict__ part_acc, float *__restrict__ part_ml, uint32_t num_heads,
                     uint32_t group, float scale_log2, const uint32_t *__restrict__ counts,
                     const uint32_t *__restrict__ mates, uint32_t pack, uint16_t *__restrict__ k_w,
                     uint16_t *__restrict__ v_w, const uint16_t *__restrict__ new_k,
                     const uint16_t *__restrict__ new_v, const uint32_t *__restrict__ new_slots,
                     uint32_t num_shared, uint32_t *__restrict__ arrivals) {
#pragma clang fp contract(off)  // the wavefronts' merge rounds as a shared pack's does
    constexpr int KK = HD / 32;
    constexpr int DT = HD / 16;
    constexpr uint32_t kTile = kBS * HD;
    __shared__ uint32_t s_col[3][16];  // per column: row, first partial, splits
    extern __shared__ float smem[];  // the wavefronts' merge (without stages)
    // The stages of a shared pack (four objects of their own, so that the
    // compiler can tell one stage's DMA from another stage's reads and waits
    // for neither); the register path's merge keeps wavefront w's
    // accumulators in stage w.
    constexpr bool kStages = W == kSharedWaves;
    constexpr uint32_t kStageBytes = kStages ? SharedStage<HD>::BYTES : 16;
    __shared__ __align__(1024) uint8_t sh0[kStageBytes];
    __shared__ __align__(1024) uint8_t sh1[kStageBytes];
    __shared__ __align__(1024) uint8_t sh2[kStageBytes];
    __shared__ __align__(1024) uint8_t sh3[kStageBytes];
    __shared__ float s_ml[kStages ? 2 * W * 16 : 1];
    __shared__ uint32_t s_last[PACKS == kNoPacks ? 1 : 64];  // who merges (arrivals)
    static_assert(!kStages || 16 * kAccStride<HD> * 4 <= kStageBytes, "merge fits a stage");

    const uint32_t item = blockIdx.x / kv_heads;
    const uint32_t kvh = blockIdx.x % kv_heads;
    // The item's record loads beside the step's count: every launched item
    // has a readable record.  The grid may be sized for more work than this
    // step has (fixed launch shapes); the step's own count is on the device.
    const u32x4 rec = *reinterpret_cast<const u32x4 *>(work + 4 * static_cast<uint64_t>(item));
    if (item >= counts[0]) return;
    const uint32_t row = rec[0];
    const uint32_t split = rec[1] & kSplitMask;
    const uint32_t *table = tables + rec[2];  // this split's block ids
    const uint32_t nk = rec[3];
    const uint64_t out_base = static_cast<uint64_t>(row) * num_heads * HD;

    if (nk == 0) {
        // The reference's empty softmax leaves the zero-filled output
        // (attention.rs:119); one work item covers such a row.
        for (uint32_t idx = threadIdx.x; idx < group * HD; idx += 64 * W)
            out[out_base + static_cast<uint64_t>(kvh) * group * HD + idx] = 0;
        return;
    }
    // Each partial was written with agent-scope stores: waits until this
    // wavefront's are done, and for the workgroup's other wavefronts.
    auto stored = []() __attribute__((always_inline)) {
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0)
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __syncthreads();
    };
    // Counts one of the `expected` items of the row whose partials start at
    // `first`, for this KV head.  True for the last, which leaves the counter
    // at zero for the next launch.
    auto count_item = [&](uint32_t first, uint32_t expected) {
        uint32_t *const count = arrivals + static_cast<uint64_t>(first) * kv_heads + kvh;
        const uint32_t before =
            __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = before + 1 == expected;
        if (last) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return last;
    };
    // This workgroup's merge of row r for its KV head's query heads.
    auto merge = [&](uint32_t r, uint32_t first, uint32_t nsplit, bool fine_row) {
        constexpr uint32_t NQ = HD / 4;
        for (uint32_t i = threadIdx.x; i < group * NQ; i += 64 * W) {
            const uint32_t qh = kvh * group + i / NQ;
            merge_row<HD, true>(part_acc, part_ml, first, nsplit, fine_row, nk, split_keys, num_heads,
                                qh, 4 * (i % NQ), out + (static_cast<uint64_t>(r) * num_heads + qh) * HD);
        }
    };
    // The end of a shared pack, when the rows' last workgroups merge: one lane
    // counts the item for each of the pack's rows (at most 64).
    auto arrive_pack = [&]() {
        stored();
        if (threadIdx.x < pack) {
            const uint32_t r = threadIdx.x == 0 ? row : mates[(pack - 1) * item + threadIdx.x - 1];
            const u32x2 info = *reinterpret_cast<const u32x2 *>(
                row_info + 2 * static_cast<uint64_t>(r == kNoMate ? row : r));
            s_last[threadIdx.x] =
                r != kNoMate && info[1] > 1 && count_item(info[0], info[1]) ? r : kNoMate;
        }
        __syncthreads();
        for (uint32_t j = 0; j < pack; ++j) {
            const uint32_t r = uniform_u32(s_last[j]);
            if (r == kNoMate) continue;
            const u32x2 info = *reinterpret_cast<const u32x2 *>(row_info + 2 * static_cast<uint64_t>(r));
            merge(r, info[0], info[1], false);
        }
    };
    if constexpr (kStages && PACKS != kNoPacks) {
        if (item < num_shared) {
            if constexpr (PACKS == kPairPacks)
                shared_split_pairs<HD, W>(k_pool, v_pool, kv_heads, kvh, item, rec, tables,
                                          row_info, split_keys, q, out, part_acc, part_ml,
                                          num_heads, group, scale_log2, mates, pack, sh0, sh1,
                                          sh2, sh3, arrivals != nullptr);
            else
                shared_split<HD, W>(k_pool, v_pool, kv_heads, kvh, item, rec, tables, row_info,
                                    split_keys, q, out, part_acc, part_ml, num_heads, group,
                                    scale_log2, mates, pack, sh0, sh1, sh2, sh3, arrivals != nullptr);
            if (arrivals) arrive_pack();
            return;
        }
    }
    // In a plan with shared packs every item with mates is one of them.
    if constexpr (PACKS != kNoPacks) pack = 1;

    const uint32_t k_begin = split * split_keys;
    const uint32_t k_end = min(nk, k_begin + split_keys);
    const uint32_t nblk = (k_end - k_begin + kBS - 1) / kBS;
    const uint32_t nchunks = (k_end - k_begin + kChunk - 1) / kChunk;
    // With new keys given, the item holding the row's last key caches it
    // and takes it from new_k / new_v (see NewKeys).
    // A fine item holds the chunks c % W == part of its split only.
    constexpr bool kFine = kStages && PACKS == kNoPacks;
    const bool fine = kFine && (rec[1] & ~kSplitMask) != 0;
    const uint32_t part = fine ? (rec[1] >> kPartShift) - 1 : 0u;
    const bool take_new = new_k != nullptr && k_end == nk && (!fine || (nchunks - 1) % W == part);
    const uint16_t *nk_row = take_new ? new_k + (static_cast<uint64_t>(row) * kv_heads + kvh) * HD : nullptr;
    const uint16_t *nv_row = take_new ? new_v + (static_cast<uint64_t>(row) * kv_heads + kvh) * HD : nullptr;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane & 15;  // MFMA column of this lane
    const int g = lane >> 4;  // lane group: keys 8g..8g+7 of a chunk

    LaneMap lm;
    {
        const int m = lane & 15;
        lm.k_off = (8 * ((m >> 2) & 1) + (m & 3)) * 32 + 8 * g;
        lm.k_hi = m >= 8;
        lm.v_off = m * kBS + 8 * (g & 1);
        lm.v_hi = g >= 2;
    }
    const uint64_t block_stride = static_cast<uint64_t>(kv_heads) * kTile;
    const uint16_t *k_head = k_pool + static_cast<uint64_t>(kvh) * kTile;
    const uint16_t *v_head = v_pool + static_cast<uint64_t>(kvh) * kTile;

    // Column h holds query head kvh*group + hh of row slot h / group: slot 0
    // is the item's own row, slot j > 0 its j-th mate (a row whose split
    // reads the same blocks); columns past the pack stay zero.  MFMA output
    // columns and the per-column softmax never mix, so a packed row gets the
    // same bits as it would alone.
    const uint32_t pslot = static_cast<uint32_t>(h) / group;
    const uint32_t hh = static_cast<uint32_t>(h) - pslot * group;
    uint32_t crow = kNoMate;
    if (pslot == 0)
        crow = row;
    else if (pslot < pack)
        crow = mates[(pack - 1) * item + pslot - 1];
    const bool head_ok = crow != kNoMate;
    const uint32_t qhead = kvh * group + hh;

    // Q^T operand: column h, dims 32*kk + 8g .. +7.
    bf16x8 qv[KK];
    {
        const uint16_t *qp =
            q + (static_cast<uint64_t>(head_ok ? crow : row) * num_heads + qhead) * HD + 8 * g;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) qv[kk] = head_ok ? load_bf16x8(qp + 32 * kk) : bf16x8{};
    }
    // The column's output place (first partial, splits), loaded now so that
    // the end of the item waits on no load; by every lane (a column without a
    // row: the item's own row's, not used), as a branch around the load ended
    // in a wait for it, and for Q, before the first chunk was asked for.
    const u32x2 cinfo =
        *reinterpret_cast<const u32x2 *>(row_info + 2 * static_cast<uint64_t>(head_ok ? crow : row));

    // The end of an item with a partial, when the row's last workgroup merges
    // (every column is this row's): the workgroup that counts the row's last
    // item for this KV head reads the partials back with agent-scope loads.
    // (No release or acquire fence: see the top of this file.)
    auto arrive = [&](uint32_t first, uint32_t nsplit, bool fine_row) {
        stored();
        if (threadIdx.x == 0)
            s_last[0] = count_item(first, fine_row ? W * (nk / split_keys) + split_states(nk % split_keys)
                                                   : nsplit);
        __syncthreads();
        if (s_last[0] != 0) merge(row, first, nsplit, fine_row);
    };

    // Block ids of chunk cc: wave-uniform, so scalar loads from the table
    // (no LDS copy, no VGPR).  Load order: mates, Q and column info, first
    // chunk, so that each wait for a value (vmcnt counts in issue order)
    // leaves the later loads in flight.  Every wave issues its first chunk,
    // a wave without one from the split's last block, so that no branch
    // leaves the compiler's wait counting unsure.
    auto load = [&](Chunk<HD> &r, uint32_t cc) {
        const uint32_t b0 = min(2 * cc, nblk - 1);
        const uint32_t p0 = table[b0];
        const uint32_t p1 = (b0 + 1 < nblk) ? table[b0 + 1] : p0;
        load_chunk<HD, NT>(r, k_head, v_head, block_stride, p0, p1, lm);
        issue_fence();
    };
    Chunk<HD> bufA, bufB;
    // This wavefront's chunks: state + (k0 + k) W for k < mine, where a fine
    // item's wavefront has run `wave` of the item's state, and another
    // item's has the whole state `wave`.
    const uint32_t state = fine ? part : static_cast<uint32_t>(wave);
    const uint32_t k0 = fine ? kSubChunks * static_cast<uint32_t>(wave) : 0u;
    const uint32_t of_state = nchunks > state ? (nchunks - state + W - 1) / W : 0;
    uint32_t mine = of_state > k0 ? of_state - k0 : 0u;
    if (fine) mine = min(mine, kSubChunks);
    auto chunk = [&](uint32_t k) { return state + (k0 + k) * W; };
    load(bufA, chunk(0));

    // Between runs the merged accumulators wait in the wavefront's stage.
    floatx4 *const run_lds = kStages ? reinterpret_cast<floatx4 *>(
        wave == 0 ? sh0 : (wave == 1 ? sh1 : (wave == 2 ? sh2 : sh3))) : nullptr;
    RunState<HD> rs;
    rs.reset();

    // A chunk computed inside the loop has a successor, so it is full: only
    // the chunks computed at the loop's exits can be the split's tail, and
    // only they carry the masking code.
    auto run = [&](Chunk<HD> &r, uint32_t cc, bool may_tail, bool first) {
        const uint32_t j0 = k_begin + cc * kChunk;
        if (may_tail && take_new && cc + 1 == nchunks)
            take_new_key<HD>(r, nk - 1 - j0, nk_row, nv_row, lane);
        const bool tail = may_tail && j0 + kChunk > k_end;
        const int nv = max(0, min(8, static_cast<int>(k_end) - static_cast<int>(j0 + 8 * g)));
        compute_chunk<HD>(r, qv, tail, nv, scale_log2, rs.m, rs.l, rs.acc, first);
    };
    // Before chunk k (even), true if it begins a run: every kSubChunks chunks.
    // (With another number of wavefronts than a pack's or a fine item's, a
    // tuning setting, a state is one run.)  The run before it ends here, ahead
    // of the next chunk's loads, whose registers it uses.
    auto new_run = [&](uint32_t k) {
        const bool first = kStages ? k % kSubChunks == 0 : k == 0;
        if constexpr (kStages)
            if (first && k != 0) rs.flush(run_lds, lane, k == kSubChunks);
        return first;
    };
    static_assert(kSubChunks % 2 == 0, "runs start at the first register buffer");

    // Two register buffers: the loads of chunk k + 1 are all issued (the
    // fence in `load`) before the first wait for chunk k, so each wavefront
    // has two chunks in flight while it waits.  The loop has one exit and
    // the last one or two chunks follow it: with an early exit inside the
    // loop, the control-flow structurizer routes that exit back through the
    // loop header, where the compiler then waits for every load in flight.
    uint32_t k = 0;
#pragma unroll 1
    for (; k + 2 < mine; k += 2) {
        const bool begins = new_run(k);
        load(bufB, chunk(k + 1));
        run(bufA, chunk(k), false, begins);
        load(bufA, chunk(k + 2));
        run(bufB, chunk(k + 1), false, false);
    }
    const bool first = new_run(k);
    if (k + 1 < mine) {
        load(bufB, chunk(k + 1));
        run(bufA, chunk(k), false, first);
        run(bufB, chunk(k + 1), true, false);
    } else if (k < mine) {
        run(bufA, chunk(k), true, first);
    }
    if constexpr (kStages) rs.finish(run_lds, lane, mine <= kSubChunks);
    float m_run = rs.m;
    float l_run = rs.l;
    floatx4 (&acc)[DT] = rs.acc;

    // Cache the new key (nothing in this launch reads its slot from the pool).
    if (take_new) {
        const uint32_t slot = new_slots[row];
        const uint64_t tile = static_cast<uint64_t>(slot / kBS) * block_stride + static_cast<uint64_t>(kvh) * kTile;
        const uint32_t t = slot % kBS;
        for (uint32_t u = threadIdx.x; u < HD / 8; u += 64 * W) {
            const uint32_t d = 8 * u;
            *reinterpret_cast<u32x4 *>(k_w + tile + (d / 32) * (kBS * 32) + t * 32 + d % 32) =
                *reinterpret_cast<const u32x4 *>(nk_row + d);
        }
        for (uint32_t d = threadIdx.x; d < HD; d += 64 * W) v_w[tile + d * kBS + t] = nv_row[d];
    }

    if constexpr (kFine) {
        if (fine) {
            // Fold the state's runs, in order, through the stages: wavefront
            // w's run sits in stage w ([DT][64] floatx4, then m and l per
            // lane), and wavefront w folds DT / W of the DT accumulators.
            uint8_t *const mine_st = wave == 0 ? sh0 : (wave == 1 ? sh1 : (wave == 2 ? sh2 : sh3));
            constexpr uint32_t ML = DT * 64 * 16;
            static_assert(ML + 2 * 64 * 4 <= kStageBytes && DT % W == 0, "a run fits a stage");
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                reinterpret_cast<floatx4 *>(mine_st)[dt * 64 + lane] = acc[dt];
            reinterpret_cast<float *>(mine_st + ML)[lane] = m_run;
            reinterpret_cast<float *>(mine_st + ML)[64 + lane] = l_run;
            __syncthreads();
            const uint32_t runs = (of_state + kSubChunks - 1) / kSubChunks;  // 1 .. W
            constexpr int DW = DT / W;
            const floatx4 *a0 = reinterpret_cast<const floatx4 *>(sh0) + (wave * DW) * 64 + lane;
            float mf = reinterpret_cast<const float *>(sh0 + ML)[lane];
            float lf = reinterpret_cast<const float *>(sh0 + ML)[64 + lane];
            floatx4 af[DW];
#pragma unroll
            for (int i = 0; i < DW; ++i) af[i] = a0[i * 64];
#pragma unroll
            for (int w = 1; w < W; ++w) {
                if (static_cast<uint32_t>(w) < runs) {
                    const uint8_t *st = w == 1 ? sh1 : (w == 2 ? sh2 : sh3);
                    floatx4 aw[DW];
#pragma unroll
                    for (int i = 0; i < DW; ++i)
                        aw[i] = reinterpret_cast<const floatx4 *>(st)[(wave * DW + i) * 64 + lane];
                    fold_state<16 * DW>(mf, lf, af, reinterpret_cast<const float *>(st + ML)[lane],
                                        reinterpret_cast<const float *>(st + ML)[64 + lane], aw);
                }
            }
            lf += __shfl_xor(lf, 16, 64);
            lf += __shfl_xor(lf, 32, 64);
            // The partial of state `part`: slot first + W split + part.
            if (head_ok) {
                const uint64_t slot = static_cast<uint64_t>(cinfo[0]) + static_cast<uint64_t>(W) * split + part;
                const uint64_t at = slot * num_heads + qhead;
                float *ap = part_acc + at * HD + 16 * DW * wave + 4 * g;
#pragma unroll
                for (int i = 0; i < DW; ++i) put_f32x4(ap + 16 * i, af[i], arrivals != nullptr);
                if (wave == 0 && g == 0) {
                    put_f32(part_ml + 2 * at, mf, arrivals != nullptr);
                    put_f32(part_ml + 2 * at + 1, lf, arrivals != nullptr);
                }
            }
            if (arrivals) arrive(uniform_u32(cinfo[0]), uniform_u32(cinfo[1]) & ~kFineRow, true);
            return;
        }
    }

    // The running sums are per lane group; the max is already per head.
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);

    if constexpr (W == 1) {
        if (head_ok) {
            const uint32_t nsplit = cinfo[1];
            const uint64_t part_base = static_cast<uint64_t>(cinfo[0] + split) * num_heads;
            if (nsplit == 1) {
                const float inv = 1.0f / l_run;
                uint16_t *op = out + static_cast<uint64_t>(crow) * num_heads * HD +
                               static_cast<uint64_t>(qhead) * HD + 4 * g;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    u32x2 packed;
                    packed[0] = f32_to_bf16_bits(acc[dt][0] * inv) |
                                (static_cast<uint32_t>(f32_to_bf16_bits(acc[dt][1] * inv)) << 16);
                    packed[1] = f32_to_bf16_bits(acc[dt][2] * inv) |
                                (static_cast<uint32_t>(f32_to_bf16_bits(acc[dt][3] * inv)) << 16);
                    *reinterpret_cast<u32x2 *>(op + 16 * dt) = packed;
                }
            } else {
                const uint64_t part = part_base + qhead;
                float *ap = part_acc + part * HD + 4 * g;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<floatx4 *>(ap + 16 * dt) = acc[dt];
                if (g == 0) {
                    part_ml[2 * part] = m_run;
                    part_ml[2 * part + 1] = l_run;
                }
            }
        }
    } else {
        // Merge the W wavefronts' (m, l, acc) through LDS.
        float *sm_m = kStages ? s_ml : smem;  // [W][16]
        float *sm_l = sm_m + W * 16;          // [W][16]
        // [W][cols][HD]: wavefront w's block at sm_acc_w(w)
        float *sm_acc = kStages ? nullptr : sm_l + W * 16;
        const uint32_t cols = pack * group;
        auto sm_acc_w = [&](int w) -> float * {
            if constexpr (kStages)
                return reinterpret_cast<float *>(w == 0 ? sh0 : (w == 1 ? sh1 : (w == 2 ? sh2 : sh3)));
            else
                return sm_acc + static_cast<uint32_t>(w) * cols * kAccStride<HD>;
        };
        if (wave == 0 && g == 0) {
            s_col[0][h] = crow;
            s_col[1][h] = cinfo[0];
            s_col[2][h] = cinfo[1];
        }
        if (head_ok) {
            if (g == 0) {
                sm_m[wave * 16 + h] = m_run;
                sm_l[wave * 16 + h] = l_run;
            }
            float *ap = sm_acc_w(wave) + h * kAccStride<HD> + 4 * g;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<floatx4 *>(ap + 16 * dt) = acc[dt];
        }
        __syncthreads();
        for (uint32_t idx = threadIdx.x; idx < cols * HD; idx += 64 * W) {
            const uint32_t col = idx / HD;
            const uint32_t d = idx % HD;
            const uint32_t r = s_col[0][col];
            if (r == kNoMate) continue;  // a short pack
            float mx = -INFINITY;
#pragma unroll
            for (int w = 0; w < W; ++w) mx = fmaxf(mx, sm_m[w * 16 + col]);
            float num = 0.0f, den = 0.0f;
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const float e = __builtin_amdgcn_exp2f(sm_m[w * 16 + col] - mx);
                num += e * sm_acc_w(w)[col * kAccStride<HD> + d];
                den += e * sm_l[w * 16 + col];
            }
            const uint32_t qh = kvh * group + (col % group);
            const uint32_t nsplit = s_col[2][col];
            if (nsplit == 1) {
                out[static_cast<uint64_t>(r) * num_heads * HD + static_cast<uint64_t>(qh) * HD + d] =
                    f32_to_bf16_bits(num / den);
            } else {
                const uint64_t part = static_cast<uint64_t>(s_col[1][col] + split) * num_heads + qh;
                put_f32(part_acc + part * HD + d, num, kStages && arrivals != nullptr);
                if (d == 0) {
                    put_f32(part_ml + 2 * part, mx, kStages && arrivals != nullptr);
                    put_f32(part_ml + 2 * part + 1, den, kStages && arrivals != nullptr);
                }
            }
        }
        if constexpr (kStages)
            if (arrivals && s_col[2][0] > 1) arrive(s_col[1][0], s_col[2][0], false);
    }
}

// Merges the split-K partials of the rows listed in reduce_rows (those with
// more than one split; rows with one split were written by the split kernel),
// where the row's last workgroup does not (no arrivals).  A wavefront is a
// workgroup and takes 64 / (HD / 4) query heads of one row, a thread four dims
// (with four such to a workgroup 65 rows of 64 heads took 5.8 us instead of
// 5.5).
template <int HD>
__global__ __launch_bounds__(64) void decode_reduce_kernel(
    const uint32_t *__restrict__ reduce_rows, const float *__restrict__ part_acc,
    const float *__restrict__ part_ml, uint16_t *__restrict__ out, uint32_t num_heads,
    const uint32_t *__restrict__ counts) {
    constexpr uint32_t NQ = HD / 4;    // dim quads of one head
    constexpr uint32_t HPW = 64 / NQ;  // heads per workgroup
    const uint32_t groups = (num_heads + HPW - 1) / HPW;
    // The row's whole record in one load (every launched row has a readable
    // one), beside the step's count.
    const u32x4 rec = *reinterpret_cast<const u32x4 *>(reduce_rows + 4 * static_cast<uint64_t>(blockIdx.x / groups));
    if (blockIdx.x / groups >= counts[1]) return;  // past this step's rows (fixed launch)
    const uint32_t qh = (blockIdx.x % groups) * HPW + threadIdx.x / NQ;
    if (qh >= num_heads) return;
    merge_row<HD, false>(part_acc, part_ml, rec[1], rec[2], false, 0, 0, num_heads, qh,
                         4 * (threadIdx.x % NQ),
                         out + (static_cast<uint64_t>(rec[0]) * num_heads + qh) * HD);
}

template <int HD, int W, bool NT, int PACKS>
hipError_t launch_split_kind(const PoolLayer &pool, const MetaView &meta, const DecodePlan &plan,
                        const uint16_t *q, uint16_t *out, uint32_t num_heads, float scale_log2,
                        hipStream_t stream, const NewKeys *nkeys) {
    const uint32_t group = num_heads / pool.kv_heads;
    const uint32_t pack = plan.pack ? plan.pack : 1;
    const uint32_t shared = plan.num_shared;
    // Shared packs: W wavefronts of up to 16 / G rows; the other items then
    // carry no mates.  (A shared pack never holds a row's new key: its blocks
    // are read by another row, so a plan with new keys has none there.)
    const uint32_t shared_tiles = plan.shared_pairs ? W / 2 : W;
    if (shared != 0 && (W != kSharedWaves || group > 16 ||
                        pack > shared_tiles * (16 / group) || plan.split_keys % kChunk != 0))
        return hipErrorInvalidValue;
    const uint32_t item_pack = shared ? 1u : pack;
    static_assert(PACKS == kNoPacks || W == kSharedWaves, "packs need the stages");
    if (plan.arrivals && (item_pack != 1 || pack > 64 || W != kSharedWaves)) return hipErrorInvalidValue;
    if (item_pack * group > 16 || (pack > 1 && plan.mates == nullptr)) return hipErrorInvalidValue;
    // With 4 wavefronts (not streaming) the merge lives in the shared-pack
    // stages (at most 16 columns of HD floats per wavefront, 8 KiB at
    // head_dim 128).
    constexpr bool kStages = W == kSharedWaves;
    const size_t smem =
        (W == 1 || kStages) ? 0
                            : (2 * W * 16 + static_cast<size_t>(W) * item_pack * group * kAccStride<HD>) * 4;
    const uint64_t grid = static_cast<uint64_t>(plan.launch_work) * pool.kv_heads;
    if (grid > 0x7fffffffull) return hipErrorInvalidValue;
    KernelTimer timer(plan.fine ? "decode_splitk_fine" : "decode_splitk", stream);
    hipLaunchKernelGGL((decode_splitk_kernel<HD, W, NT, PACKS>), dim3(static_cast<uint32_t>(grid)),
                       dim3(64 * W), smem, stream, pool.k, pool.v, pool.kv_heads, meta.tables,
                       plan.work, plan.row_info,
                       plan.split_keys, q, out, plan.part_acc, plan.part_ml, num_heads, group,
                       scale_log2, plan.counts, plan.mates, pack, pool.k, pool.v,
                       nkeys ? nkeys->k : nullptr, nkeys ? nkeys->v : nullptr,
                       nkeys ? nkeys->slots : nullptr, shared, plan.arrivals);
    return hipGetLastError();
}

template <int HD, int W, bool NT>
hipError_t launch_split(const PoolLayer &pool, const MetaView &meta, const DecodePlan &plan,
                        const uint16_t *q, uint16_t *out, uint32_t num_heads, float scale_log2,
                        hipStream_t stream, const NewKeys *nkeys) {
    if constexpr (W == kSharedWaves) {
        if (plan.num_shared != 0 && plan.shared_pairs)
            return launch_split_kind<HD, W, NT, kPairPacks>(pool, meta, plan, q, out, num_heads,
                                                            scale_log2, stream, nkeys);
        if (plan.num_shared != 0)
            return launch_split_kind<HD, W, NT, kSinglePacks>(pool, meta, plan, q, out, num_heads,
                                                              scale_log2, stream, nkeys);
    }
    return launch_split_kind<HD, W, NT, kNoPacks>(pool, meta, plan, q, out, num_heads, scale_log2,
                                                  stream, nkeys);
}

template <int HD>
hipError_t launch_hd(const PoolLayer &pool, const MetaView &meta, const DecodePlan &plan,
                     const uint16_t *q, uint16_t *out, uint32_t num_heads, float scale_log2,
                     int waves, hipStream_t stream, const NewKeys *nkeys) {
    hipError_t err;
    const bool nt = plan.streaming;
#define VO_SPLIT(Wv)                                                                            \
    (nt ? launch_split<HD, Wv, true>(pool, meta, plan, q, out, num_heads, scale_log2, stream,  \
                                     nkeys)                                                  \
        : launch_split<HD, Wv, false>(pool, meta, plan, q, out, num_heads, scale_log2, stream, \
                                      nkeys))
    switch (waves) {
        case 1: err = VO_SPLIT(1); break;
        case 2: err = VO_SPLIT(2); break;
        case 8: err = VO_SPLIT(8); break;
        default: err = VO_SPLIT(4); break;
    }
#undef VO_SPLIT
    if (err != hipSuccess || plan.launch_reduce == 0 || plan.arrivals) return err;
    constexpr uint32_t kHeadsPerGroup = 64 / (HD / 4);
    const uint64_t grid = static_cast<uint64_t>(plan.launch_reduce) *
                          ((num_heads + kHeadsPerGroup - 1) / kHeadsPerGroup);
    if (grid > 0x7fffffffull) return hipErrorInvalidValue;
    KernelTimer timer("decode_reduce", stream);
    hipLaunchKernelGGL((decode_reduce_kernel<HD>), dim3(static_cast<uint32_t>(grid)), dim3(64),
                       0, stream, plan.reduce_rows, plan.part_acc, plan.part_ml, out, num_heads,
                       plan.counts);
    return hipGetLastError();
}

}  // namespace

bool decode_mfma_supported(uint32_t head_dim, uint32_t block_size, uint32_t group) {
    return (head_dim == 64 || head_dim == 128) && block_size == kBS && group >= 1 && group <= 16;
}

hipError_t launch_decode_mfma(const PoolLayer &pool, const MetaView &meta,
                              const DecodePlan &plan, const uint16_t *q, uint16_t *out,
                              uint32_t num_heads, float scale, int waves_per_group,
                              hipStream_t stream, const NewKeys *new_keys) {
    if (plan.launch_work == 0) return hipSuccess;
    // New keys need exactly the plan's items (not a fixed launch's grid).
    if (new_keys && plan.launch_work != plan.num_work) return hipErrorInvalidValue;
    if (plan.split_keys == 0 || plan.split_keys % kChunk != 0 || plan.split_keys > kMaxSplitKeys)
        return hipErrorInvalidValue;
    const float scale_log2 = scale * 1.4426950408889634f;
    switch (pool.head_dim) {
        case 64:
            return launch_hd<64>(pool, meta, plan, q, out, num_heads, scale_log2, waves_per_group,
                                 stream, new_keys);
        case 128:
            return launch_hd<128>(pool, meta, plan, q, out, num_heads, scale_log2,
                                  waves_per_group, stream, new_keys);
        default:
            return hipErrorInvalidValue;
    }
}

}  // namespace kernels
}  // namespace vo
