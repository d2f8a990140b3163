// Token + position embedding for gfx950.
//
// Reference behaviour: FINAL_CLEAN_CODE/src/kernels/embedding.cu (gather,
// in-place position add, float-atomic scatter-add backward) and the CPU
// loops of NEW_code/tests/test_embedding.cu:16-41.
//
// Forward: a wave per few token rows, or per row chunk where there are few
// tokens, W-wide vector copies; the fused variant
// writes table[id] + pos[t] in one pass (one fp32 add, so bit-identical to
// the reference's gather followed by its in-place add).
//
// Token backward, deterministic and bit-identical to the CPU loop, which
// adds grad rows into grad_table in increasing token position: one kernel,
// no workspace (emb_bwd_owner_kernel below).  The ids are split into classes
// and each class belongs to a few workgroups, every one of which collects
// the positions of the class's ids from the whole id vector and sorts them by
// id in LDS.  Each element (table row, column) has exactly one workgroup that
// updates it in a call, in position order: a row's columns are shared out
// over the class's workgroups where the id is frequent or the class's list
// does not fit LDS at once, and go to one workgroup otherwise.
// Position backward: one thread per (t, column vector) adds grad_out[b, t]
// for b = 0, 1, ... in order onto grad_pos[t]; the fused token + position
// backward does the same sums inside the token kernel's workgroups.
#include <type_traits>

#include "mi_common.hpp"

namespace mi {

namespace {

constexpr int kRowWaves = 4;   // token rows per workgroup

// ---------------------------------------------------------------------------
// Forward
// ---------------------------------------------------------------------------
// Each wave gathers R consecutive token rows: the R ids are read first,
// then the loads of all R rows (table and position, NQ vectors per lane per
// row at a time) are issued before any row is stored, so that R row gathers
// are in flight per wave instead of one behind each id load.
template <int W, bool POS, int R, int NQ>
__global__ __launch_bounds__(kRowWaves * kWave) void emb_fwd_kernel(
    const float* __restrict__ table, const float* __restrict__ pos, const int* __restrict__ tokens,
    float* __restrict__ out, int batch_seq, int seq, int dim, int vocab) {
    const int lane = threadIdx.x & (kWave - 1);
    const int i0 = (blockIdx.x * kRowWaves + static_cast<int>(threadIdx.x / kWave)) * R;
    if (i0 >= batch_seq) return;  // wave-uniform
    const int nv = dim / W;
    int id[R];
    bool ok[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = i0 + r < batch_seq ? i0 + r : batch_seq - 1;
        id[r] = tokens[i];
        ok[r] = i0 + r < batch_seq && (vocab <= 0 || (id[r] >= 0 && id[r] < vocab));
    }
    for (int j0 = lane; j0 < nv; j0 += NQ * kWave) {
        fvec<W> v[R][NQ];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float* src = table + static_cast<size_t>(ok[r] ? id[r] : 0) * dim;
            const float* p = POS ? pos + static_cast<size_t>((i0 + r) % seq) * dim : nullptr;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int j = j0 + q * kWave;
                // Table rows are gathered with the non-temporal hint: in the
                // config-2 step (forward after the previous backward) it
                // measured 65.1 -> 64.1 us, although a forward repeated
                // alone, which finds the 154 MB table in the last-level
                // cache, is faster without it (15.9 us).
                v[r][q] = (ok[r] && j < nv) ? sload<W>(src, j) : vzero<W>();
                if constexpr (POS) {
                    if (j < nv && i0 + r < batch_seq) {
                        const fvec<W> t = vload<W>(p, j);
#pragma unroll
                        for (int e = 0; e < W; ++e) v[r][q].v[e] = v[r][q].v[e] + t.v[e];
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (i0 + r >= batch_seq) break;  // wave-uniform
            float* dst = out + static_cast<size_t>(i0 + r) * dim;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int j = j0 + q * kWave;
                // streamed out: measured 20.9 -> 16.0 us at config 2
                if (j < nv) sstore<W>(dst, j, v[r][q]);
            }
        }
    }
}

// The gather for few tokens, where the form above leaves most of the chip idle
// and each wave waits for one row chunk after another (16 tokens of 1600
// columns: one workgroup, 6.2 us): a wave takes one row's chunk of 64 vectors,
// so every load of the call is in flight at once (512 tokens of 320, fwd +
// bwd, 16.8 -> 8.8 us).
template <int W, bool POS>
__global__ __launch_bounds__(kRowWaves * kWave) void emb_fwd_chunk_kernel(
    const float* __restrict__ table, const float* __restrict__ pos, const int* __restrict__ tokens,
    float* __restrict__ out, int batch_seq, int seq, int dim, int vocab, int chunks) {
    const int lane = threadIdx.x & (kWave - 1);
    const int u = blockIdx.x * kRowWaves + static_cast<int>(threadIdx.x / kWave);
    const int i = u / chunks;
    if (i >= batch_seq) return;  // wave-uniform
    const int j = (u - i * chunks) * kWave + lane;
    const int nv = dim / W;
    const int id = tokens[i];
    const bool ok = vocab <= 0 || (id >= 0 && id < vocab);
    if (j >= nv) return;
    fvec<W> t = vzero<W>();
    if constexpr (POS) t = vload<W>(pos + static_cast<size_t>(i % seq) * dim, j);
    fvec<W> v = ok ? sload<W>(table + static_cast<size_t>(id) * dim, j) : vzero<W>();
    if constexpr (POS) {
#pragma unroll
        for (int e = 0; e < W; ++e) v.v[e] = v.v[e] + t.v[e];
    }
    sstore<W>(out + static_cast<size_t>(i) * dim, j, v);
}

// embeddings[b, t, :] += pos[t, :], one wave per row.
template <int W>
__global__ __launch_bounds__(kRowWaves * kWave) void pos_add_kernel(const float* __restrict__ pos,
                                                                    float* __restrict__ emb,
                                                                    int rows, int seq, int dim) {
    const int lane = threadIdx.x & (kWave - 1);
    const int i = blockIdx.x * kRowWaves + static_cast<int>(threadIdx.x / kWave);
    if (i >= rows) return;
    const int nv = dim / W;
    const float* p = pos + static_cast<size_t>(i % seq) * dim;
    float* dst = emb + static_cast<size_t>(i) * dim;
#pragma unroll 4
    for (int j = lane; j < nv; j += kWave) {
        fvec<W> v = vload<W>(dst, j);
        const fvec<W> q = vload<W>(p, j);
#pragma unroll
        for (int e = 0; e < W; ++e) v.v[e] = v.v[e] + q.v[e];
        vstore<W>(dst, j, v);
    }
}

// grad_pos[t, j] += grad_out[b, t, j] for b = 0..batch-1 in order.
template <int W>
__global__ __launch_bounds__(256) void pos_bwd_kernel(const float* __restrict__ g,
                                                      float* __restrict__ gpos, int batch,
                                                      int seq, int dim) {
    const int nv = dim / W;
    const long long idx = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= static_cast<long long>(seq) * nv) return;
    const int t = static_cast<int>(idx / nv);
    const int j = static_cast<int>(idx % nv);
    const size_t row_stride = static_cast<size_t>(seq) * nv;  // in vectors
    const size_t base = static_cast<size_t>(t) * nv + j;
    fvec<W> acc = vload<W>(gpos, base);
    int b = 0;
    // Latency-bound at small seq * dim (a thread per vector, few threads):
    // 8 rows per round trip instead of 4.
    for (; b + 8 <= batch; b += 8) {
        fvec<W> q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) q[u] = vload<W>(g, base + (b + u) * row_stride);
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int e = 0; e < W; ++e) acc.v[e] = acc.v[e] + q[u].v[e];
    }
    for (; b < batch; ++b) {
        const fvec<W> q = vload<W>(g, base + b * row_stride);
#pragma unroll
        for (int e = 0; e < W; ++e) acc.v[e] = acc.v[e] + q.v[e];
    }
    vstore<W>(gpos, base, acc);
}

// ---------------------------------------------------------------------------
// Token backward, owner-computes form.  The valid ids are split into K (a
// power of two) classes, id % K, and each class belongs to S workgroups.
// Every workgroup reads the whole id vector (4 bytes per token, served from
// L2, against 3 KB of grad row per token) and keeps the positions of its
// class's ids, in position order, in an LDS list, which is sorted by id in
// LDS, stably, so that each id's entries form a run in increasing position.
// Runs of at least kHeavy rows are added by the S workgroups together, each
// its own slice of the columns (add_heavy); a shorter run is added by one wave
// of one of them (one load of the table row, the run's grad rows in order,
// one store).  Every element of a table row therefore receives its grad rows
// in increasing token position, as in the CPU loop, and the result is
// bit-identical whichever workgroup or wave adds it.
//
// What bounds it depends on the ids.  Uniform over a large vocabulary (16384
// tokens, D = 768, V = 50257: fwd + bwd 53.4 us, 54.2 with one workgroup per
// class and every run on one wave): the random 3 KB rows, behind the scan and
// the sort, during which only the position rows stream (the token backward
// takes 26.9 us, and 12.6 with rows of 64 columns).  Frequencies of text on the
// same shape: the longest runs, 67 us against 202 us when one wave added each
// (a memory round trip per two rows of a 466-row run).  A few characters (32 x
// 256 tokens of 65 ids, D = 512): 23 us against 287 us.
// ---------------------------------------------------------------------------
constexpr int kOwnWaves = 8;
constexpr int kOwnThreads = kOwnWaves * kWave;   // 512
constexpr int kOwnPer = 32;                      // ids per thread per pass
constexpr int kOwnPerSmall = 8;                  // the same for small token counts
constexpr int kOwnCap = 2048;                    // list entries per window
constexpr int kOwnTake = 2;                      // sorted entries per claim
constexpr int kOwnMaxGrid = 512;                 // workgroups, at most
// Neighbouring values, token backward in us, 64 or 768 columns of 50257 ids:
//   kOwnLog2S 1 / 2 / 3    16384 tokens x 768, text 54.3 / 36.1 / 33.1, uniform 26.2 /
//                          26.5 / 28.1; 16384 x 64 uniform 10.8 / 12.1 / 13.9
//   kOwnTokens 4 / 8 / 16  1000 x 768 uniform 5.9 / 6.9 / 8.9, text 8.6 / 10.1 / 11.5;
//                          2048 x 64 uniform 6.1 / 5.5 / 6.4, x 768 text 10.8 / 9.8 / 10.2
//   kHeavy 8 / 16 / 32     2048 x 64 text 11.5 / 8.8 / 8.8; 512 x 768 of 65 ids, text 10.3 /
//                          10.2 / 12.1, uniform 10.7 / 7.4 / 7.4
constexpr int kOwnList = 256;                    // list entries a class should have, at most
constexpr int kOwnLog2S = 2;                     // log2 of the workgroups that share a class
constexpr int kOwnTokens = 8;                    // tokens per workgroup, at least
constexpr int kHeavy = 16;                       // rows of a run that the class's workgroups share
// Vectors per thread per staged batch of a long run (32 KB of LDS with 16-byte
// vectors, 16 KB with scalars).
template <int W>
constexpr int heavy_vecs() {
    return W == 4 ? 4 : 8;
}
constexpr int kSlotBits = 11;                    // bits of a list slot in a key
static_assert(kOwnCap == 1 << kSlotBits, "a list slot fits its bits");
static_assert(kOwnCap % kHeavy == 0, "s_heavy holds every long run of a list");
constexpr int kRankMax = 128;                    // longest list sorted by rank, and
constexpr int kRankWide = 384;                   // the same in place of two digits or more

// Position gradient fused into the owner kernel (POS): the workgroups also
// share out the seq * nv position column vectors, one per thread per round;
// each is grad_pos[t, j] + grad_out[0, t, j] + grad_out[1, t, j] + ... in
// increasing b, the order of pos_bwd_kernel.  The old values and the first
// kPosPre batch rows of a thread's first vector are requested before the
// id scan and summed after it, so that they stream from HBM while the
// workgroup scans ids and builds its list (HBM is otherwise idle then); the
// partial sums wait in LDS, and the remaining rows are added after the
// token gradient.
constexpr int kPosPre = 7;   // batch rows in flight across the id scan, at most
constexpr int kPosChunk = 5; // batch rows per group of loads afterwards

// 128 VGPRs at most, so that two 8-wave workgroups fit on a CU.
template <int W, int NCH, int PER, bool POS>
__global__ __launch_bounds__(kOwnThreads) __attribute__((amdgpu_waves_per_eu(4))) void
emb_bwd_owner_kernel(int n, int vocab, int dim, int batch, int seq, int cfg,
                     const int* __restrict__ ids, const float* __restrict__ g,
                     float* __restrict__ table, float* __restrict__ gpos) {
    constexpr int kSpan = kOwnThreads * PER;       // positions per pass
    constexpr int kHeavyU = heavy_vecs<W>();
    constexpr unsigned kBins = kOwnThreads * kHeavyU * W / kOwnWaves;  // counts kept in s_stage
    constexpr int kBinBits = 31 - __builtin_clz(kBins);
    static_assert(kBins == 1u << kBinBits && kBins % kOwnThreads == 0, "digits of whole bits");
    // Grad rows per group of loads in a short run: as many as the registers
    // of NCH column vectors per lane leave room for.
    constexpr int kBatch = NCH == 1 ? 8 : NCH == 2 ? 4 : 2;
    // The list: keys and positions, [0] in position order, sorted in [srt]
    // (with room for the padding that the rank sort reads).  A key is the
    // id's number within the class (id / K) with the list slot in its low
    // bits, where it fits 32 bits so (`slots`; without a vocabulary bound the
    // slot is put in once the list is known); no two keys are then equal, and
    // their order is the stable order by id.
    __shared__ __align__(16) unsigned s_keyb[2][kOwnCap + 16];
    __shared__ int s_posb[2][kOwnCap];
    __shared__ int s_wsum[kOwnWaves];
    __shared__ int s_count[3];  // runs claimed, long runs, short runs
    int& s_next = s_count[0];
    int& s_nheavy = s_count[1];
    int& s_nlight = s_count[2];
    __shared__ int s_heavy[kOwnCap / kHeavy], s_hlen[kOwnCap / kHeavy];  // long runs
    __shared__ __align__(16) float s_stage[kOwnThreads * kHeavyU * W];  // their staged rows
    unsigned* const s_key = s_keyb[0];
    int* const s_pos = s_posb[0];
    int srt = 1;  // buffer that holds the sorted list
    __shared__ fvec<W> s_pacc[POS ? kOwnThreads : 1];  // first position rows, summed
    const int lane = threadIdx.x & (kWave - 1);
    // Uniform over the wave; readfirstlane lets the compiler see that, so
    // branches on it are scalar branches, not exec-masked ones.
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
    // cfg packs log2 K and log2 S (one preloaded argument).
    const int log2k = cfg & 31;
    const int log2s = cfg >> 5;
    const int nblk = 1 << (log2k + log2s);
    const unsigned k = blockIdx.x & ((1u << log2k) - 1u);
    const int part = static_cast<int>(blockIdx.x >> log2k);
    const int nv = dim / W;
    // An id of class k: rotating id ^ k right by log2 K leaves id / K, and a
    // value of at least 2^(32 - log2 K) for the ids of other classes, so one
    // unsigned compare with the number of this class's valid ids tests the
    // class, the vocabulary bound and the sign together.
    const unsigned vlim = vocab > 0 ? static_cast<unsigned>(vocab) : 0x80000000u;
    const unsigned qlim = vlim > k ? ((vlim - 1u - k) >> log2k) + 1u : 0u;
    auto number = [&](int id) __attribute__((always_inline)) {
        const unsigned x = static_cast<unsigned>(id) ^ k;
        return __builtin_amdgcn_alignbit(x, x, static_cast<unsigned>(log2k));
    };
    constexpr unsigned kSlotNum = (1u << (32 - kSlotBits)) - 1u;  // numbers below it leave room for a slot
    const bool slots = qlim <= kSlotNum;
    int kshift = slots ? kSlotBits : 0;
    auto key_of = [&](unsigned num, int slot) __attribute__((always_inline)) {
        return slots ? (num << kSlotBits) | static_cast<unsigned>(slot) : num;
    };
    // The class number of a sorted entry, and the id it stands for.
    auto num_at = [&](int e) __attribute__((always_inline)) { return s_keyb[srt][e] >> kshift; };
    auto id_of = [&](unsigned num) __attribute__((always_inline)) {
        return static_cast<size_t>((num << log2k) | k);
    };
    // This workgroup's column vectors of the long runs: slice `part` of S,
    // whole 128-byte lines each (the last ones may be empty).
    constexpr int kLine = 32 / W;
    const int svec = (((nv + (1 << log2s) - 1) >> log2s) + kLine - 1) / kLine * kLine;
    const int cbeg = part * svec;
    const int cend = cbeg + svec < nv ? cbeg + svec : nv;

    // Short runs: a workgroup adds whole rows ([lb, le) is [0, nv)) of the ids
    // that are its own within the class.  Where a class fills its list more
    // than once, an id's run may be long in one and short in the next, so
    // every workgroup of the class then keeps to its column slice for the
    // short runs too: each part of a table row has one workgroup that
    // updates it, in list order.
    bool sliced = false;
    int lb = 0;
    int le = nv;

    const unsigned long long below = (1ull << lane) - 1ull;

    // acc += the grad rows of sorted-list entries from, from + 1, ... while
    // they carry class number `num` (none if entry `from` does not), in list
    // order, for the column vectors c0 + lane + q * 64.
    auto add_entries = [&](unsigned num, int from, int L, int c0, fvec<W>(&acc)[NCH]) __attribute__((always_inline)) {
        for (int off = from;; off += kWave) {
            const int e = off + lane;
            const bool same = e < L && num_at(e) == num;
            const int pos_l = same ? s_posb[srt][e] : 0;
            const unsigned long long m = __ballot(same);
            const int cnt =
                (~m == 0ull) ? kWave : (__ffsll(static_cast<unsigned long long>(~m)) - 1);
            for (int u0 = 0; u0 < cnt; u0 += kBatch) {
                fvec<W> v[kBatch][NCH];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    const int src = u0 + u < cnt ? u0 + u : 0;
                    const float* grow = g + static_cast<size_t>(__shfl(pos_l, src, kWave)) * dim;
#pragma unroll
                    for (int q = 0; q < NCH; ++q) {
                        const int j = c0 + lane + q * kWave;
                        v[u][q] = (u0 + u < cnt && j < le) ? vload<W>(grow, j) : vzero<W>();
                    }
                }
#pragma unroll
                for (int u = 0; u < kBatch; ++u)
                    if (u0 + u < cnt) {
#pragma unroll
                        for (int q = 0; q < NCH; ++q)
#pragma unroll
                            for (int x = 0; x < W; ++x) acc[q].v[x] = acc[q].v[x] + v[u][q].v[x];
                    }
            }
            if (cnt < kWave) break;
        }
    };

    // Adds the run starting at sorted-list entry s0 (entries s0, s0 + 1, ...
    // with the id of s0, in position order) onto that id's table row.
    auto add_run = [&](int s0, int L) __attribute__((always_inline)) {
        const unsigned num = num_at(s0);
        float* row = table + id_of(num) * dim;
        for (int c0 = lb; c0 < le; c0 += NCH * kWave) {
            fvec<W> acc[NCH];
#pragma unroll
            for (int q = 0; q < NCH; ++q) {
                const int j = c0 + lane + q * kWave;
                acc[q] = j < le ? vload<W>(row, j) : vzero<W>();
            }
            add_entries(num, s0, L, c0, acc);
#pragma unroll
            for (int q = 0; q < NCH; ++q) {
                const int j = c0 + lane + q * kWave;
                if (j < le) vstore<W>(row, j, acc[q]);
            }
        }
    };

    // Adds the runs starting at sorted-list entries sa and sb together: the
    // two table rows and the first grad row of each run are requested at
    // once; the rest of each run (if any) follows.
    auto add_pair = [&](int sa, int sb, int L) __attribute__((always_inline)) {
        const unsigned na = num_at(sa);
        const unsigned nb = num_at(sb);
        float* ra = table + id_of(na) * dim;
        float* rb = table + id_of(nb) * dim;
        const float* ga = g + static_cast<size_t>(s_posb[srt][sa]) * dim;
        const float* gb = g + static_cast<size_t>(s_posb[srt][sb]) * dim;
        for (int c0 = lb; c0 < le; c0 += NCH * kWave) {
            fvec<W> A[NCH], B[NCH];
            {
                fvec<W> GA[NCH], GB[NCH];
#pragma unroll
                for (int q = 0; q < NCH; ++q) {
                    const int j = c0 + lane + q * kWave;
                    const bool ok = j < le;
                    A[q] = ok ? vload<W>(ra, j) : vzero<W>();
                    B[q] = ok ? vload<W>(rb, j) : vzero<W>();
                    GA[q] = ok ? vload<W>(ga, j) : vzero<W>();
                    GB[q] = ok ? vload<W>(gb, j) : vzero<W>();
                }
#pragma unroll
                for (int q = 0; q < NCH; ++q)
#pragma unroll
                    for (int x = 0; x < W; ++x) {
                        A[q].v[x] = A[q].v[x] + GA[q].v[x];
                        B[q].v[x] = B[q].v[x] + GB[q].v[x];
                    }
            }
            add_entries(na, sa + 1, L, c0, A);
            add_entries(nb, sb + 1, L, c0, B);
#pragma unroll
            for (int q = 0; q < NCH; ++q) {
                const int j = c0 + lane + q * kWave;
                if (j < le) {
                    vstore<W>(ra, j, A[q]);
                    vstore<W>(rb, j, B[q]);
                }
            }
        }
    };

    // Adds the long runs (s_heavy / s_hlen) onto their table rows with the
    // whole workgroup.  One wave adding such a run alone waits for a memory
    // round trip per kBatch rows, which for the frequent ids of text
    // (hundreds of rows per id) took longer than everything else; here the
    // workgroup streams the rows through LDS, 512 * kHeavyU vectors per batch
    // with two batches in flight in registers, and each thread adds the
    // staged rows of one column in list order, so the sums are the ones a
    // single wave would form, bit for bit.  The S workgroups of the class each
    // add their own column slice, in chunks of 2^lcv vectors.  The batches of
    // all chunks of all runs follow each other without a gap (run by run, a
    // run of one batch took 5 us).
    auto add_heavy = [&](int nheavy) __attribute__((always_inline)) {
        int lcv = 3;
        while (lcv < (W == 4 ? 6 : 8) && (1 << lcv) < cend - cbeg) ++lcv;
        const int cv = 1 << lcv;
        const int cw = cv * W;                                // columns per chunk
        const int rpp = kOwnThreads >> lcv;                   // rows per vector of a thread
        const int rb = rpp * kHeavyU;                         // rows per batch
        const int vec = threadIdx.x & (cv - 1);
        const int r0 = static_cast<int>(threadIdx.x) >> lcv;
        const int col = static_cast<int>(threadIdx.x);
        // Where the requests and the sums are: run h (entries s0 .. s0 + cnt),
        // chunk from column vector c0, row b of the run.
        struct At {
            int h, s0, cnt, c0, b;
            float* row;
        };
        auto enter = [&](At& a) __attribute__((always_inline)) {
            a.s0 = __builtin_amdgcn_readfirstlane(s_heavy[a.h]);
            a.cnt = __builtin_amdgcn_readfirstlane(s_hlen[a.h]);
            a.row = table + id_of(static_cast<unsigned>(
                                __builtin_amdgcn_readfirstlane(static_cast<int>(num_at(a.s0))))) *
                                dim;
            a.c0 = cbeg;
            a.b = 0;
        };
        auto advance = [&](At& a) __attribute__((always_inline)) {
            a.b += rb;
            if (a.b >= a.cnt) {
                a.b = 0;
                a.c0 += cv;
                if (a.c0 >= cend) {
                    ++a.h;
                    if (a.h < nheavy) enter(a);
                }
            }
        };
        At rq, su;
        rq.h = 0;
        enter(rq);
        su = rq;
        struct Batch {
            fvec<W> v[kHeavyU];
            float old;
        };
        // Loads are clamped into the run and the slice (past the last batch
        // they repeat rows of the last run); only rows and columns in range
        // are added.
        auto request = [&](Batch& d) __attribute__((always_inline)) {
            const int j = rq.c0 + vec < cend ? rq.c0 + vec : cend - 1;
#pragma unroll
            for (int u = 0; u < kHeavyU; ++u) {
                const int r = rq.b + u * rpp + r0;
                const int p = s_posb[srt][rq.s0 + (r < rq.cnt ? r : rq.cnt - 1)];
                d.v[u] = vload<W>(g + static_cast<size_t>(p) * dim, j);
            }
            const int oc = rq.c0 * W + col;
            d.old = rq.row[oc < cend * W ? oc : cend * W - 1];
            advance(rq);
        };
        // A wave alone on its SIMD issues an instruction every 4 to 8 cycles,
        // so the sums, one LDS read and one dependent add per row, are most
        // of a batch's time; the row pitch is a constant so that the reads
        // need no address arithmetic (30 cycles a row with it, 20 without).
        // Only the last group may be partial (its reads stay in the batch).
        auto sum_rows = [](float a, const float* p, int rows, auto pitch) __attribute__((always_inline)) {
            constexpr int kPitch = decltype(pitch)::value;
            for (int r = 0; r < rows; r += 16, p += 16 * kPitch) {
                float x[16];
#pragma unroll
                for (int q = 0; q < 16; ++q) x[q] = p[q * kPitch];
                if (r + 16 <= rows) {
#pragma unroll
                    for (int q = 0; q < 16; ++q) a = a + x[q];
                } else {
#pragma unroll
                    for (int q = 0; q < 16; ++q) a = r + q < rows ? a + x[q] : a;
                }
            }
            return a;
        };
        float cur = 0.0f;
        auto consume_batch = [&](Batch& d) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < kHeavyU; ++u)
                *reinterpret_cast<fvec<W>*>(&s_stage[((u * rpp + r0) * cv + vec) * W]) = d.v[u];
            cur = su.b == 0 ? d.old : cur;
            request(d);
            __syncthreads();
            if (su.h < nheavy) {
                if (col < cw) {
                    const int left = su.cnt - su.b;
                    const int rows = left < rb ? left : rb;
                    const float* p = s_stage + col;
                    switch (lcv) {
                        case 3: cur = sum_rows(cur, p, rows, std::integral_constant<int, 8 * W>{}); break;
                        case 4: cur = sum_rows(cur, p, rows, std::integral_constant<int, 16 * W>{}); break;
                        case 5: cur = sum_rows(cur, p, rows, std::integral_constant<int, 32 * W>{}); break;
                        default:
                            if constexpr (W == 4) {
                                cur = sum_rows(cur, p, rows, std::integral_constant<int, 64 * W>{});
                            } else {
                                if (lcv == 6)
                                    cur = sum_rows(cur, p, rows, std::integral_constant<int, 64>{});
                                else if (lcv == 7)
                                    cur = sum_rows(cur, p, rows, std::integral_constant<int, 128>{});
                                else
                                    cur = sum_rows(cur, p, rows, std::integral_constant<int, 256>{});
                            }
                    }
                    const int oc = su.c0 * W + col;
                    if (su.b + rb >= su.cnt && oc < cend * W) su.row[oc] = cur;
                }
                advance(su);
            }
            __syncthreads();
        };
        // In this order: swapped by the scheduler, the first batch's wait
        // became a wait for both, in every trip of the loop.  All batches every
        // time: with a batch conditional, the compiler waited for all
        // outstanding loads before each one.
        Batch A, B;
        request(A);
        __builtin_amdgcn_sched_barrier(0);
        request(B);
        __builtin_amdgcn_sched_barrier(0);
        do {
            consume_batch(A);
            consume_batch(B);
        } while (su.h < nheavy);
    };

    // Sorts list entries [0, L) by id, stably: short lists by rank, four
    // threads an entry, longer ones by counting, digit by digit of kBinBits
    // bits, low digit first; one digit holds a class of up to kBins ids.  Ranks
    // grow with the square of the list (11 us at 450 entries), a digit costs 1
    // to 2 us however long it is, hence the lines (64 columns, us, ranks up to
    // 64 / 128 / 192: 8192 uniform ids of 50257, lists of 64 on average, 11.4 /
    // 10.2 / 10.2; 16384 of 50257, lists of 128, 12.4 / 12.5 / 12.1, of 5000 11.0 /
    // 11.0 / 11.1; 2048 with the frequencies of 65 letters 8.3 / 8.2 / 9.3; two
    // digits: 24576 of 151936, ranks up to 192 / 256 22.0 / 19.6).  One bit a
    // pass, which calls without a vocabulary bound took for every list, cost 1
    // us a bit (16384 ids of 50257, no bound: 16.9 us, 12.7 now; 16 ids: 10.8, 4.7
    // now).
    //
    // Runs of at least kHeavy rows are added by the class's workgroups
    // together, by column slices; of the shorter runs a workgroup takes those
    // whose id / K mod S is its number, and its waves share them out through
    // an LDS counter.  Each run is added in position order whoever adds it,
    // so the result does not depend on the assignment.
    auto process = [&](int L) __attribute__((always_inline)) {
        if (threadIdx.x < 3) s_count[threadIdx.x] = 0;
        // No number of the list is above `top`.  Where the vocabulary bound
        // says little, the list does, and where the keys have no slot for
        // want of a bound they get one now.
        unsigned top = L > 1 ? qlim - 1u : 0u;
        if (!slots) kshift = 0;
        if (L > 1 && (!slots || (top >= kBins && L > kRankWide))) {
            unsigned any = 0;
            for (int i = static_cast<int>(threadIdx.x); i < L; i += kOwnThreads) any |= s_key[i];
            any = wave_or(any);
            if (lane == 0) s_wsum[wave] = static_cast<int>(any);
            __syncthreads();
            any = 0;
#pragma unroll
            for (int w = 0; w < kOwnWaves; ++w) any |= static_cast<unsigned>(s_wsum[w]);
            top = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(any))) >> kshift;
            if (!slots && top < kSlotNum) {
                for (int i = static_cast<int>(threadIdx.x); i < L; i += kOwnThreads)
                    s_key[i] = (s_key[i] << kSlotBits) | static_cast<unsigned>(i);
                kshift = kSlotBits;
            }
        }
        if (top == 0) {
            srt = 0;  // one id at most: sorted as it is
        } else if (L <= (top < kBins || kshift == 0 ? kRankMax : kRankWide)) {
            srt = 1;
            if (threadIdx.x < 16) s_key[L + threadIdx.x] = 0xffffffffu;
            __syncthreads();
            const int sub = static_cast<int>(threadIdx.x) & 3;
            for (int i0 = 0; i0 < L; i0 += kOwnThreads / 4) {
                const int i = i0 + (static_cast<int>(threadIdx.x) >> 2);
                if (i0 + wave * (kWave / 4) >= L) break;  // wave-uniform
                const unsigned me = s_key[i < L ? i : 0];
                int r = 0;
                if (kshift != 0) {
#pragma unroll 4
                    for (int j = 4 * sub; j < L; j += 16) {
                        const uint4 o = *reinterpret_cast<const uint4*>(&s_key[j]);
                        r += (o.x < me) + (o.y < me) + (o.z < me) + (o.w < me);
                    }
                } else {
                    // Keys without the slot: equal ones in list order.
                    for (int j = 4 * sub; j < L; j += 16) {
                        const uint4 o = *reinterpret_cast<const uint4*>(&s_key[j]);
                        r += (o.x < me || (o.x == me && j < i)) +
                             (o.y < me || (o.y == me && j + 1 < i)) +
                             (o.z < me || (o.z == me && j + 2 < i)) +
                             (o.w < me || (o.w == me && j + 3 < i));
                    }
                }
                r += __shfl_xor(r, 1, kWave);
                r += __shfl_xor(r, 2, kWave);
                if (i < L) {
                    if (sub == 0) s_keyb[1][r] = me;
                    if (sub == 1) s_posb[1][r] = s_pos[i];
                }
            }
        } else {
            // Wave w holds entries w * span + [0, span) in groups of 64.  A
            // group's lanes find the lanes of the same digit from one ballot
            // per bit; an entry's place among its digit's entries is the
            // wave's count before the group plus the equal lanes below it.
            // The counts of all waves, summed over the waves and then over
            // the digits, give every (wave, digit) its first slot.
            constexpr int kQ = kOwnCap / kOwnThreads;
            const int span = (L + kOwnThreads - 1) / kOwnThreads * kWave;
            int* const cnt = reinterpret_cast<int*>(s_stage);  // [wave][kBins]
            int lo = kshift;
            const int hi = kshift + 32 - __builtin_clz(top);
            srt = 0;
#pragma unroll 1
            for (; lo < hi; lo += kBinBits) {
                const int nbits = hi - lo < kBinBits ? hi - lo : kBinBits;
                // Thread t takes the digits t * kPer + [0, kPer) of those there
                // are (no number has a bit from hi up); waves past them have
                // nothing to clear or add.
                constexpr int kPer = kBins / kOwnThreads;
                int* const mine = cnt + static_cast<int>(threadIdx.x) * kPer;
                const bool some = threadIdx.x * kPer < (1u << nbits);
                if (some) {
#pragma unroll
                    for (int b = 0; b < kPer; ++b)
#pragma unroll
                        for (int w = 0; w < kOwnWaves; ++w) mine[w * kBins + b] = 0;
                }
                __syncthreads();
                auto digit = [&](unsigned key) __attribute__((always_inline)) {
                    return (key >> lo) & (kBins - 1u);
                };
                unsigned me[kQ];
                int at[kQ];
#pragma unroll
                for (int q = 0; q < kQ; ++q) {
                    if (q * kWave >= span) break;  // uniform
                    const int i = wave * span + q * kWave + lane;
                    const bool ok = i < L;
                    me[q] = ok ? s_keyb[srt][i] : 0u;
                    const unsigned num = digit(me[q]);
                    unsigned long long same = __ballot(ok);
                    for (int b = 0; b < nbits; ++b) {
                        const bool bit = ((num >> b) & 1u) != 0;
                        const unsigned long long m = __ballot(bit);
                        same &= bit ? m : ~m;
                    }
                    int* const c = &cnt[wave * kBins + num];
                    const int upto = ok ? *c : 0;
                    at[q] = upto + __popcll(same & below);
                    // The counts pass between the wave's lanes: every lane has
                    // read its count before the lowest equal lane updates it,
                    // and the update is made before the next group reads.
                    wave_order();
                    if (ok && (same & below) == 0ull) *c = upto + __popcll(same);
                    wave_order();
                }
                __syncthreads();
                int bsum = 0;
                if (some) {
#pragma unroll
                    for (int b = 0; b < kPer; ++b)
#pragma unroll
                        for (int w = 0; w < kOwnWaves; ++w) bsum += mine[w * kBins + b];
                }
                int upto = bsum;  // inclusive sum over the wave's lanes
#pragma unroll
                for (int o = 1; o < kWave; o *= 2) {
                    const int v = __shfl_up(upto, o, kWave);
                    upto += lane >= o ? v : 0;
                }
                if (lane == kWave - 1) s_wsum[wave] = upto;
                __syncthreads();
                int run = upto - bsum;
#pragma unroll
                for (int w = 0; w < kOwnWaves; ++w) run += w < wave ? s_wsum[w] : 0;
                if (some) {
#pragma unroll
                    for (int b = 0; b < kPer; ++b)
#pragma unroll
                        for (int w = 0; w < kOwnWaves; ++w) {
                            const int v = mine[w * kBins + b];
                            mine[w * kBins + b] = run;
                            run += v;
                        }
                }
                __syncthreads();
#pragma unroll
                for (int q = 0; q < kQ; ++q) {
                    if (q * kWave >= span) break;
                    const int i = wave * span + q * kWave + lane;
                    if (i < L) {
                        const int to = cnt[wave * kBins + digit(me[q])] + at[q];
                        s_keyb[srt ^ 1][to] = me[q];
                        s_posb[srt ^ 1][to] = s_posb[srt][i];
                    }
                }
                srt ^= 1;
                __syncthreads();
            }
        }
        __syncthreads();
        // The runs: long ones into s_heavy, this workgroup's short ones into
        // the key buffer that the sort has left free.
        unsigned* const s_light = s_keyb[srt ^ 1];
        for (int i0 = 0; i0 < L; i0 += kOwnThreads) {
            const int i = i0 + static_cast<int>(threadIdx.x);
            const unsigned me = i < L ? num_at(i) : 0u;
            const bool start = i < L && (i == 0 || num_at(i - 1) != me);
            const bool heavy = start && i + kHeavy <= L && num_at(i + kHeavy - 1) == me;
            if (heavy) {
                int lo = i + kHeavy, hi = L;  // end of the run in [lo, hi]
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (num_at(mid) == me)
                        lo = mid + 1;
                    else
                        hi = mid;
                }
                const int slot = atomicAdd(&s_nheavy, 1);
                s_heavy[slot] = i;
                s_hlen[slot] = lo - i;
            }
            const bool light =
                start && !heavy &&
                (sliced || static_cast<int>(me & ((1u << log2s) - 1u)) == part);
            const unsigned long long m = __ballot(light);
            int at = 0;
            if (lane == 0 && m != 0) at = atomicAdd(&s_nlight, static_cast<int>(__popcll(m)));
            at = __shfl(at, 0, kWave);
            if (light) s_light[at + __popcll(m & below)] = static_cast<unsigned>(i);
        }
        __syncthreads();
        if (cbeg < cend) {
            const int nheavy = __builtin_amdgcn_readfirstlane(s_nheavy);
            if (nheavy > 0) add_heavy(nheavy);
        }
        const int nlight = s_nlight;
        for (;;) {
            int e = 0;
            if (lane == 0) e = atomicAdd(&s_next, kOwnTake);
            e = __shfl(e, 0, kWave);
            if (e >= nlight) break;
            if (kOwnTake == 2 && e + 1 < nlight)
                add_pair(static_cast<int>(s_light[e]), static_cast<int>(s_light[e + 1]), L);
            else
                add_run(static_cast<int>(s_light[e]), L);
        }
    };

    // Position gradient, first round: requests issued now, summed below.
    const long long pvec = POS ? static_cast<long long>(seq) * nv : 0;   // position vectors
    const long long pstride = static_cast<long long>(nblk) * kOwnThreads;
    // A thread's first position vector, below kOwnMaxGrid * kOwnThreads = 2^18:
    // 32 bits.  Held as a 64-bit value it was spilled to scratch, and its
    // reload waited for every outstanding load.
    const int pv0 = static_cast<int>(blockIdx.x) * kOwnThreads + wave * kWave + lane;
    const size_t bstride = static_cast<size_t>(seq) * nv;                // vectors per batch row
    // PRE batch rows of the first position vector are requested across the
    // id scan (7 for 2-3 column vectors per lane, 4 for one: more spills
    // registers in the scan).
    constexpr int PRE = !POS ? 0 : NCH == 1 ? 4 : kPosPre;
    constexpr int NPQ = PRE > 0 ? PRE : 1;
    // Adds batch rows b0, b0 + 1, ... of position vector pv onto acc, in
    // order, and stores the total.  Whole groups load unconditionally: with
    // each load under a uniform branch the compiler may put waits between a
    // group's loads (token + position backward, 500 x 64 tokens of 768: 114 us so,
    // 88 now).
    auto pos_rest = [&](long long pv, int b0, fvec<W> acc) __attribute__((always_inline)) {
        int b = b0;
        for (; b + kPosChunk <= batch; b += kPosChunk) {
            fvec<W> q[kPosChunk];
#pragma unroll
            for (int u = 0; u < kPosChunk; ++u) q[u] = sload<W>(g, (b + u) * bstride + pv);
#pragma unroll
            for (int u = 0; u < kPosChunk; ++u)
#pragma unroll
                for (int x = 0; x < W; ++x) acc.v[x] = acc.v[x] + q[u].v[x];
        }
        if (b < batch) {
            fvec<W> q[kPosChunk - 1];
#pragma unroll
            for (int u = 0; u < kPosChunk - 1; ++u)
                q[u] = b + u < batch ? sload<W>(g, (b + u) * bstride + pv) : vzero<W>();
#pragma unroll
            for (int u = 0; u < kPosChunk - 1; ++u)
                if (b + u < batch)
#pragma unroll
                    for (int x = 0; x < W; ++x) acc.v[x] = acc.v[x] + q[u].v[x];
        }
        vstore<W>(gpos, pv, acc);
    };
    // The position vectors after a thread's first one (pv0 + pstride, ...).
    auto pos_others = [&]() __attribute__((always_inline)) {
        for (long long pv = pv0 + pstride; pv < pvec; pv += pstride)
            pos_rest(pv, 0, vload<W>(gpos, pv));
    };

    // One scan of kSpan positions of the id vector: this class's ids are
    // appended to the list, behind the `filled` entries that it holds, if they
    // all fit; `total` says how many there are.  The first scan is a separate
    // instantiation (FIRST) so that the position registers live only inside
    // it.  This lambda and those it calls are inlined: an out-of-line call
    // keeps the captured locals in scratch memory.
    int filled = 0, total = 0, before = 0;
    unsigned wpos = 0;
    const unsigned un = static_cast<unsigned>(n);
    auto scan = [&](unsigned base, auto first_tag) __attribute__((always_inline)) {
        constexpr bool first = decltype(first_tag)::value && PRE > 0;
        [[maybe_unused]] fvec<W> pacc, pq[NPQ];
        // Wave w reads positions base + w * PER * 64 + [0, PER * 64), load e
        // of lane l position 64 e + l of it: list order is load order, then
        // lane order, and every load instruction of the wave reads 256
        // contiguous bytes.
        wpos = base + static_cast<unsigned>(wave) * PER * kWave;
        int my[PER];
        // The choice is uniform over the wave and no load sits under a
        // per-lane branch, so the waits that follow count these loads
        // exactly: with per-lane branches the compiler waited for all but
        // one of the position loads issued below before the first id was
        // tested, which serialised them with the scan.
        if (wpos + PER * kWave <= un) {
#pragma unroll
            for (int e = 0; e < PER; ++e) my[e] = ids[wpos + e * kWave + lane];
        } else {
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                const unsigned p = wpos + e * kWave + lane;
                const int v = ids[p < un ? p : un - 1u];
                my[e] = p < un ? v : -1;
            }
        }
        if constexpr (first) {
            // Issued after the id loads: loads complete in issue order, so
            // the scan can use its ids while these are still in flight.
            // Unconditional loads, issued back to back on every lane: rows
            // past the batch are clamped to its last row and lanes past the
            // last position vector to that vector, and neither is added.
            // With the loads under a per-lane branch the compiler's wait
            // counts for the ids below had to allow for a path without
            // them, and each id group then waited for one more of these.
            const long long pvc = pv0 < pvec ? pv0 : pvec - 1;
            pacc = vload<W>(gpos, static_cast<size_t>(pvc));
#pragma unroll
            for (int u = 0; u < PRE; ++u)
                pq[u] = sload<W>(g, static_cast<size_t>(u < batch ? u : batch - 1) * bstride +
                                        static_cast<size_t>(pvc));
        }
        // List slots in position order: the wave's matches are counted, its
        // first slot comes from the other waves' counts, and a second look at
        // the ids (in registers, three instructions each) writes them.
        int wtot = 0;
#pragma unroll
        for (int e = 0; e < PER; ++e) wtot += __popcll(__ballot(number(my[e]) < qlim));
        if (lane == 0) s_wsum[wave] = wtot;
        __syncthreads();
        before = 0;
        total = 0;
#pragma unroll
        for (int w = 0; w < kOwnWaves; ++w) {
            const int t = s_wsum[w];
            before += w < wave ? t : 0;
            total += t;
        }
        before = __builtin_amdgcn_readfirstlane(before);
        total = __builtin_amdgcn_readfirstlane(total);
        __syncthreads();  // s_wsum is rewritten later
        const bool fits = filled + total <= kOwnCap;
        if (fits && wtot > 0) {
            int at = filled + before;
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                const unsigned num = number(my[e]);
                const bool ok = num < qlim;
                const unsigned long long m = __ballot(ok);
                if (m != 0) {
                    const int slot = at + __popcll(m & below);
                    if (ok) {
                        s_key[slot] = key_of(num, slot);
                        s_pos[slot] = static_cast<int>(wpos + e * kWave + lane);
                    }
                    at += __popcll(m);
                }
            }
        }
        if (fits) filled += total;
        if constexpr (first) {
            if (pv0 < pvec) {
#pragma unroll
                for (int u = 0; u < PRE; ++u)
                    if (u < batch)
#pragma unroll
                        for (int x = 0; x < W; ++x) pacc.v[x] = pacc.v[x] + pq[u].v[x];
                s_pacc[threadIdx.x] = pacc;  // finished after the token gradient
            }
        }
        return fits;
    };
    // Entries [w0, w0 + kOwnCap) of the span last scanned into the empty
    // list, the ids read again one at a time (rare: the list was full, or one
    // span holds more of the class's ids than a list does).
    auto refill = [&](int w0) __attribute__((always_inline)) {
        int at = before;
#pragma unroll 1
        for (int e = 0; e < PER; ++e) {
            const unsigned p = wpos + e * kWave + lane;
            const unsigned num = number(p < un ? ids[p] : -1);
            const bool ok = num < qlim;
            const unsigned long long m = __ballot(ok);
            const int slot = at + __popcll(m & below) - w0;
            if (ok && slot >= 0 && slot < kOwnCap) {
                s_key[slot] = key_of(num, slot);
                s_pos[slot] = static_cast<int>(p);
            }
            at += __popcll(m);
        }
    };
    // Scan spans until the list is full or the ids are done, then add the
    // list's runs.  All of this is uniform over the workgroup, and the same
    // for every workgroup of a class.
    bool over = !scan(0u, std::true_type{});
    unsigned base = 0;
    int w0 = 0;
    for (bool done = false; !done;) {
        bool flush = true;
        if (over && filled == 0) {
            refill(w0);
            filled = total - w0 < kOwnCap ? total - w0 : kOwnCap;
            w0 += filled;
            over = w0 < total;
            flush = over;
        } else if (!over) {
            if (un - base > static_cast<unsigned>(kSpan)) {
                base += kSpan;
                over = !scan(base, std::false_type{});
                w0 = 0;
                flush = false;
            } else {
                done = true;
            }
        }
        if (flush && filled > 0) {
            if (!done) {
                sliced = true;
                lb = cbeg;
                le = cend;
            }
            __syncthreads();
            process(filled);
            __syncthreads();
            filled = 0;
        }
    }
    // The rest of the position sums follow the token gradient: the table-row
    // updates start as soon as the list is built (config-2 step 58.8 ->
    // 58.3 us against finishing the position sums first).
    if constexpr (POS) {
        if (pv0 < pvec) pos_rest(pv0, PRE, s_pacc[threadIdx.x]);
        pos_others();
    }
}

#ifndef MI_EMB_ROWS
#define MI_EMB_ROWS 4
#endif
// Token rows per wave in the forward gather.  Config 2 step (V = 50257,
// D = 768, 16384 tokens): 1 row 60.1 us, 2 rows 60.7, 4 rows 59.1, 8 rows 63.8.
constexpr int kEmbRows = MI_EMB_ROWS;

constexpr long long kChunkWaves = 8192;

// Forward gather launch: kEmbRows rows per wave, NQ = vectors per lane per
// row at a time (just enough for the row, at most 4).
template <bool POS>
void launch_emb_fwd(const float* table, const float* pos, const int* tokens, float* out,
                    int batch_seq, int seq, int dim, int vocab, hipStream_t st) {
    const bool v4 = dim % 4 == 0 && aligned16(table) && aligned16(out) && (!POS || aligned16(pos));
    const int nv = v4 ? dim / 4 : dim;
    const int nq = nv <= kWave ? 1 : nv <= 2 * kWave ? 2 : nv <= 3 * kWave ? 3 : 4;
    // Up to kChunkWaves waves of one chunk each (2 x 500 tokens of 768: fwd +
    // bwd 23.2 -> 19.1 us); past that (8 x 1024 of 512) the two forms are
    // within 4% and the rows form reads each id once per row.
    const long long chunks = (nv + kWave - 1) / kWave;
    if (batch_seq * chunks <= kChunkWaves) {
        const dim3 cgrid(static_cast<unsigned>((batch_seq * chunks + kRowWaves - 1) / kRowWaves));
        if (v4)
            hipLaunchKernelGGL((emb_fwd_chunk_kernel<4, POS>), cgrid, dim3(kRowWaves * kWave), 0,
                               st, table, pos, tokens, out, batch_seq, seq, dim, vocab,
                               static_cast<int>(chunks));
        else
            hipLaunchKernelGGL((emb_fwd_chunk_kernel<1, POS>), cgrid, dim3(kRowWaves * kWave), 0,
                               st, table, pos, tokens, out, batch_seq, seq, dim, vocab,
                               static_cast<int>(chunks));
        return;
    }
    const long long waves = (static_cast<long long>(batch_seq) + kEmbRows - 1) / kEmbRows;
    const dim3 grid(static_cast<unsigned>((waves + kRowWaves - 1) / kRowWaves)),
        block(kRowWaves * kWave);
#define MI_FWD_CASE(WW, QQ)                                                                     \
    hipLaunchKernelGGL((emb_fwd_kernel<WW, POS, kEmbRows, QQ>), grid, block, 0, st, table, pos, \
                       tokens, out, batch_seq, seq, dim, vocab)
    switch ((v4 ? 10 : 0) + nq) {
        case 11: MI_FWD_CASE(4, 1); break;
        case 12: MI_FWD_CASE(4, 2); break;
        case 13: MI_FWD_CASE(4, 3); break;
        case 14: MI_FWD_CASE(4, 4); break;
        case 1: MI_FWD_CASE(1, 1); break;
        case 2: MI_FWD_CASE(1, 2); break;
        case 3: MI_FWD_CASE(1, 3); break;
        default: MI_FWD_CASE(1, 4); break;
    }
#undef MI_FWD_CASE
}

// One launch of the owner kernel: a grid of 2^want workgroups, at least
// kOwnTokens tokens each, as K = 2^log2k id classes of S = 2^log2s
// workgroups.  S is 4, less where a class would then have more than kOwnList
// tokens on average (a longer list takes longer to sort), and more where the
// vocabulary has fewer ids than that leaves classes (characters, bytes).  With
// kOwnList 256 / 192, token backward of 32000 tokens of 768 columns: text
// frequencies over 50257 ids 74.1 / 96.9 us, uniform ids 52.3 / 50.4 (52.0 with
// one workgroup per class), uniform over 151936 56.8 / 55.0 (54.5 so).  The
// position gradient (POS) needs 16-byte alignment of grad_pos as well for the
// vector path.
template <bool POS>
void launch_owner(const float* grad_out, const int* tokens, float* grad_table, float* grad_pos,
                  int batch_seq, int batch, int seq, int dim, int vocab, hipStream_t st) {
    const bool v4 = dim % 4 == 0 && aligned16(grad_out) && aligned16(grad_table) &&
                    (!POS || aligned16(grad_pos));
    int want = 0;
    while ((2 << want) <= kOwnMaxGrid && (2ll << want) * kOwnTokens <= batch_seq) ++want;
    int log2k = want > kOwnLog2S ? want - kOwnLog2S : 0;
    while (log2k < want && (batch_seq >> log2k) > kOwnList) ++log2k;
    if (vocab > 0)
        while (log2k > 0 && (1 << log2k) > vocab) --log2k;
    const int log2s = want - log2k;
    const dim3 grid(1u << want), block(kOwnThreads);
    const int cfg = log2k | (log2s << 5);
    const int nv = v4 ? dim / 4 : dim;
    // Column vectors per lane held at once, at most 3: the fewest that cover
    // the row in as few column chunks.
    const int chunks = (nv + 3 * kWave - 1) / (3 * kWave);
    const int nch = (nv + chunks * kWave - 1) / (chunks * kWave);
    const bool small = batch_seq <= kOwnThreads * kOwnPerSmall;
#define MI_OWNER_LAUNCH(WW, NN, PP)                                                            \
    hipLaunchKernelGGL((emb_bwd_owner_kernel<WW, NN, PP, POS>), grid, block, 0, st, batch_seq, \
                       vocab, dim, batch, seq, cfg, tokens, grad_out, grad_table, grad_pos)
#define MI_OWNER_CASE(WW, NN)                       \
    if (small)                                      \
        MI_OWNER_LAUNCH(WW, NN, kOwnPerSmall);      \
    else                                            \
        MI_OWNER_LAUNCH(WW, NN, kOwnPer)
    switch ((v4 ? 10 : 0) + nch) {
        case 11: MI_OWNER_CASE(4, 1); break;
        case 12: MI_OWNER_CASE(4, 2); break;
        case 13: MI_OWNER_CASE(4, 3); break;
        case 1: MI_OWNER_CASE(1, 1); break;
        case 2: MI_OWNER_CASE(1, 2); break;
        default: MI_OWNER_CASE(1, 3); break;
    }
#undef MI_OWNER_CASE
#undef MI_OWNER_LAUNCH
}

}  // namespace
}  // namespace mi

using namespace mi;

extern "C" {

size_t mi_embedding_backward_workspace(int) { return 0; }

int mi_embedding_forward(const float* table, const int* tokens, float* out, int batch_seq,
                         int dim, int vocab, void* stream) {
    const char* name = "mi_embedding_forward";
    if (batch_seq < 0 || dim <= 0)
        return set_error(MI_ERR_INVALID_ARG, "%s: batch_seq=%d dim=%d", name, batch_seq, dim);
    if (batch_seq == 0) return MI_OK;
    if (!table || !tokens || !out) return set_error(MI_ERR_INVALID_ARG, "%s: NULL", name);
    launch_emb_fwd<false>(table, nullptr, tokens, out, batch_seq, 1, dim, vocab,
                          to_stream(stream));
    return check_launch(name);
}

int mi_embedding_pos_forward(const float* table, const float* pos_table, const int* tokens,
                             float* out, int batch, int seq, int dim, int vocab, void* stream) {
    const char* name = "mi_embedding_pos_forward";
    if (batch < 0 || seq <= 0 || dim <= 0)
        return set_error(MI_ERR_INVALID_ARG, "%s: batch=%d seq=%d dim=%d", name, batch, seq, dim);
    const long long bt = static_cast<long long>(batch) * seq;
    if (bt == 0) return MI_OK;
    if (bt > INT32_MAX) return set_error(MI_ERR_INVALID_ARG, "%s: batch*seq too large", name);
    if (!table || !pos_table || !tokens || !out)
        return set_error(MI_ERR_INVALID_ARG, "%s: NULL", name);
    launch_emb_fwd<true>(table, pos_table, tokens, out, static_cast<int>(bt), seq, dim, vocab,
                         to_stream(stream));
    return check_launch(name);
}

int mi_pos_embedding_forward(const float* pos_table, float* embeddings, int batch, int seq,
                             int dim, void* stream) {
    const char* name = "mi_pos_embedding_forward";
    if (batch < 0 || seq <= 0 || dim <= 0)
        return set_error(MI_ERR_INVALID_ARG, "%s: batch=%d seq=%d dim=%d", name, batch, seq, dim);
    const long long rows = static_cast<long long>(batch) * seq;
    if (rows == 0) return MI_OK;
    if (rows > INT32_MAX) return set_error(MI_ERR_INVALID_ARG, "%s: batch*seq too large", name);
    if (!pos_table || !embeddings) return set_error(MI_ERR_INVALID_ARG, "%s: NULL", name);
    const dim3 grid(static_cast<unsigned>((rows + kRowWaves - 1) / kRowWaves)),
        block(kRowWaves * kWave);
    hipStream_t st = to_stream(stream);
    if (dim % 4 == 0 && aligned16(pos_table) && aligned16(embeddings))
        hipLaunchKernelGGL(pos_add_kernel<4>, grid, block, 0, st, pos_table, embeddings,
                           static_cast<int>(rows), seq, dim);
    else
        hipLaunchKernelGGL(pos_add_kernel<1>, grid, block, 0, st, pos_table, embeddings,
                           static_cast<int>(rows), seq, dim);
    return check_launch(name);
}

int mi_pos_embedding_backward(const float* grad_out, float* grad_pos_table, int batch, int seq,
                              int dim, void* stream) {
    const char* name = "mi_pos_embedding_backward";
    if (batch < 0 || seq <= 0 || dim <= 0)
        return set_error(MI_ERR_INVALID_ARG, "%s: batch=%d seq=%d dim=%d", name, batch, seq, dim);
    if (batch == 0) return MI_OK;
    if (!grad_out || !grad_pos_table) return set_error(MI_ERR_INVALID_ARG, "%s: NULL", name);
    hipStream_t st = to_stream(stream);
    const bool v4 = dim % 4 == 0 && aligned16(grad_out) && aligned16(grad_pos_table);
    const long long threads = static_cast<long long>(seq) * (v4 ? dim / 4 : dim);
    const dim3 grid(static_cast<unsigned>((threads + 255) / 256));
    if (v4)
        hipLaunchKernelGGL(pos_bwd_kernel<4>, grid, dim3(256), 0, st, grad_out, grad_pos_table,
                           batch, seq, dim);
    else
        hipLaunchKernelGGL(pos_bwd_kernel<1>, grid, dim3(256), 0, st, grad_out, grad_pos_table,
                           batch, seq, dim);
    return check_launch(name);
}

int mi_embedding_backward(const float* grad_out, const int* tokens, float* grad_table,
                          int batch_seq, int dim, int vocab, void* stream) {
    const char* name = "mi_embedding_backward";
    if (batch_seq < 0 || dim <= 0)
        return set_error(MI_ERR_INVALID_ARG, "%s: batch_seq=%d dim=%d", name, batch_seq, dim);
    if (batch_seq == 0) return MI_OK;
    if (!grad_out || !tokens || !grad_table) return set_error(MI_ERR_INVALID_ARG, "%s: NULL", name);
    launch_owner<false>(grad_out, tokens, grad_table, nullptr, batch_seq, 0, 1, dim, vocab,
                        to_stream(stream));
    return check_launch(name);
}

int mi_embedding_pos_backward(const float* grad_out, const int* tokens, float* grad_table,
                              float* grad_pos_table, int batch, int seq, int dim, int vocab,
                              void* stream) {
    const char* name = "mi_embedding_pos_backward";
    if (batch < 0 || seq <= 0 || dim <= 0)
        return set_error(MI_ERR_INVALID_ARG, "%s: batch=%d seq=%d dim=%d", name, batch, seq, dim);
    const long long bt = static_cast<long long>(batch) * seq;
    if (bt == 0) return MI_OK;
    if (bt > INT32_MAX) return set_error(MI_ERR_INVALID_ARG, "%s: batch*seq too large", name);
    if (!grad_out || !tokens || !grad_table || !grad_pos_table)
        return set_error(MI_ERR_INVALID_ARG, "%s: NULL", name);
    launch_owner<true>(grad_out, tokens, grad_table, grad_pos_table, static_cast<int>(bt), batch,
                       seq, dim, vocab, to_stream(stream));
    return check_launch(name);
}

}  // extern "C"
