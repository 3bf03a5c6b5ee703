// Device code for LEAP decode attention on gfx950 (CDNA4, wave64).
//
// One launch performs the whole attention block of one layer step for one or
// more sequences (the reference's FloatTransformer.cpp:396-662):
//   - RoPE of q: every workgroup rotates the q heads of its KV group with the
//     fp32 table row `pos` (FloatTransformer.cpp:404-494);
//   - the KV append: the workgroup whose chunk holds `pos` rotates k_new,
//     stores k_new / v_new into cache[layer][pos] and uses them in registers;
//   - split-K flash decoding over the positions [0, pos]: a workgroup owns one
//     (sequence, KV head, chunk of positions); its waves stream
//     interleaved sub-tiles of K and V rows straight into registers with
//     128-bit buffer loads, and every wave serves all q heads of the KV group
//     from those registers: GQA score (:496-630), online softmax (running
//     max / sum, :216-238) and the weighted-V accumulation (:634-661);
//   - the merge of the chunk partials by arrival counters in L2: each chunk
//     writes an unnormalised partial (o, max, sum) and counts itself in; the
//     last arrival folds.  Up to 40 chunks, every chunk counts into the final
//     counter and its last arrival folds all records as one batch of loads.
//     When every CU runs two workgroups of the launch, a CU receives its data
//     in issue order, so the first-dispatched half of a group's chunks
//     finishes earlier than the rest: that half folds in sub-groups of
//     kSubGroup while the stream runs, and the second half counts straight
//     into the final counter, whose last arrival folds the second half's
//     chunk records and the first half's sub-group records in one level.
//     Otherwise (more chunks, or 4 KiB records) a two-level tree: sub-groups
//     of kSubGroup consecutive chunks fold into one record each, and the last
//     sub-group to finish folds those.  No fold pulls more than about 80 KiB
//     through one CU.
// A batch whose groups do not cut evenly over the CUs runs the same body over
// equal runs of rows that may end one sequence and begin the next (the flat
// launches, decode_attention_flat_kernel).
//
// XCD placement.  Workgroups are dealt to the XCDs round-robin by workgroup
// id, so id % 8 names the XCD (the same holds within a 1-, 2- or 4-XCD
// partition).  The grid is numbered so that every workgroup of one
// (sequence, KV head) group has id % 8 == group % 8: the whole group runs on
// one XCD and shares that XCD's L2.  Partials, the arrival counter and the
// merge reads therefore stay in L2 (stores drain to L2, the atomic executes in
// L2, merge loads bypass only L1) instead of travelling to memory.  Within a
// group, consecutive chunks are neighbouring ids, and with eight KV heads a
// row's eight head slices are requested by neighbouring workgroups.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace leap {

constexpr int kWave = 64;
constexpr int kMaxChunks = 512;           // split-K chunks per (sequence, KV head)
constexpr int kSubGroup = 8;              // chunks per first-level merge
constexpr int kCtrStride = 32;            // ints between arrival counters: one 128-byte line each
constexpr int kFinalMax = 40;            // records of a one-level fold (the asymmetric merge's 36 at 64 chunks)
constexpr int kXcds = 8;                  // XCDs of an MI355X
constexpr int kGiveUp = 1 << 20;          // added to a final counter by a fold helper that stopped waiting
constexpr int kHelpPolls = 16384;         // a fold helper's polls of the final counter (a few ms)
constexpr int kHelpMinRecords = 32;       // records from which two workgroups share a final fold
constexpr int kSc1 = 16;                  // cache policy sc1 (device scope): miss in L1, read L2
constexpr int kNt = 2;                    // cache policy nt: streamed once (the K/V rows of a step)

// Division by a launch constant d >= 1 of numerators n < 2^31, as a
// multiply-high and a shift (Granlund and Montgomery, "Division by Invariant
// Integers using Multiplication", PLDI 1994, section 4, figure 4.1): with
// s = ceil(log2 d) and m = floor(2^32 (2^s - d) / d) + 1 < 2^32,
// n / d = (mulhi(n, m) + n) >> s, and mulhi(n, m) + n < 2n does not wrap.
// The host computes (m, s) once per launch, so that the prologue's
// quotients (workgroup id to chunk and group, group to sequence, positions
// to chunks) take three scalar instructions each instead of a reciprocal
// on the vector unit, its move back to a scalar register and the
// correction steps, which lie on the path to the first loads.
struct FastDiv {
    uint32_t m, s;
};
__host__ __device__ constexpr FastDiv make_fastdiv(uint32_t d)
{
    uint32_t s = 0;
    while ((1ull << s) < d) s++;
    return FastDiv{(uint32_t)((((1ull << s) - d) << 32) / d + 1), s};
}
__host__ __device__ __forceinline__ uint32_t fast_div(uint32_t n, FastDiv f)
{
#ifdef __HIP_DEVICE_COMPILE__
    return (__umulhi(n, f.m) + n) >> f.s;
#else
    return (uint32_t)((((uint64_t)n * f.m) >> 32) + n) >> f.s;
#endif
}

// Partial records per head of a launch with grid_chunks chunks per sequence:
// one per chunk, then one per first-level sub-group.
__host__ __device__ constexpr int records_per_head(int grid_chunks)
{
    return grid_chunks + (grid_chunks + kSubGroup - 1) / kSubGroup;
}

// Counter words per (sequence, KV head) of a launch with grid_chunks chunks
// per sequence: the final counter, then one per first-level sub-group, each
// on its own 128-byte line.  Every counter is zero between launches, so
// launches of different sizes may lay them out differently.
__host__ __device__ constexpr int counters_per_group(int grid_chunks)
{
    return (1 + (grid_chunks + kSubGroup - 1) / kSubGroup) * kCtrStride;
}

// ---- flat launches (decode_attention_flat_kernel) ----------------------------
//
// A batch's groups (sequence, KV head) rarely cut into equal chunks that are
// a whole number per CU: lengths differ, and the sequences need not divide
// the CUs.  A flat launch has n_wg workgroups per XCD, all resident, and cuts
// the XCD's rows, its groups ("items": item i of XCD x is group 8 i + x) laid
// end to end, into n_wg runs of equal length.  A run that reaches over an
// item's end is two segments or more, each a chunk of its item.  Starting a
// segment costs a workgroup about as much as kFlatSegmentRows rows (its q,
// first rows, combine and merge lie in series), so an item counts that many
// rows more than it has, ahead of its first: a run that holds a start takes
// fewer rows.
// Measured against 0, 32, 64, 96, 192 and 256 rows over ragged batches of
// 2-64 sequences of 550-4400 rows at the shapes of Llama-3-8B, Llama-3-70B
// and TinyLlama: 128 is the fastest or within 2% in the mean (0: +5-8%).
constexpr int kFlatSegmentRows = 128;
constexpr int kFlatMinRun = 64;          // rows of a run at least: one pass of 4 waves
constexpr int kFlatMaxItems = 64;        // items per XCD at most: one lane each
// A run of a large batch holds thousands of rows.  Every kFlatFlushPasses
// passes a wave adds its output accumulators to sums in LDS and its row sums
// to a second register, and starts them anew: a sum over n passes is n / 4
// additions of sums over 4, where a uniform chunk of a ragged batch is one
// chain of about 12 passes (and one of a large equal batch, of up to all of
// them).  Error against 64 bits, 64 sequences of 512-8192 rows of Llama-3-8B's
// heads (runs of 8700 rows): 4.7e-7 without, 4.0e-7 at 16 passes, 3.6e-7 at 4
// (uniform chunks of 768 rows: 3.8e-7); over seven batches of the three shapes
// the mean is 0.99 of the uniform chunks'.  At 2 and 1 passes it is 0.98 and
// TinyLlama's batches are 6-9% slower.  Equal scores, whose sum rounds the same
// way at every addition (n 2^-26 at the worst), six sequences of 30000-90000
// rows: 2.0e-6 with the row sums of a run in one chain, 7.8e-7 now (TinyLlama's
// batches 0.7% slower for it, the others as fast).
constexpr int kFlatFlushPasses = 4;

// Segment (workgroup w, item i) has record w + i among its XCD's: along the
// rows w and i only grow, and one of them grows from a segment to the next,
// so an item's segments have consecutive records.  After the n_wg + n_items
// of them come the records of first-level sub-groups (flat_sub_record: the
// item's first, from its first segment's record).
__host__ __device__ constexpr int flat_sub_record(int n_wg, int n_items, int rec0, int item)
{
    return n_wg + n_items + rec0 / kSubGroup + item;
}
__host__ __device__ constexpr int flat_records(int n_wg, int n_items)
{
    return flat_sub_record(n_wg, n_items, n_wg + n_items, n_items) + 1;
}

// Rows [begin, end) of item `item`, whose sequence is at position pos, as
// chunk lc of n_local of them; rec0: the item's first chunk's record.
struct FlatSegment {
    int item, pos, lc, n_local, begin, end, rec0;
};
// The segment of workgroup w's run [at, stop) in the item that counts rows
// [item_begin, item_end), start_rows of them ahead of its first row; an empty
// one (begin == end) if the run ends before that row.
__host__ __device__ __forceinline__ FlatSegment flat_segment(int w, int run, int at, int stop, int item,
                                                             int item_begin, int item_end, int start_rows)
{
    const int row0 = item_begin + start_rows;  // the item's first row
    const int b = at > row0 ? at : row0, e = stop < item_end ? stop : item_end;
    if (e <= b) return FlatSegment{item, 0, 0, 0, 0, 0, 0};
    const int w_first = (int)((unsigned)row0 / (unsigned)run), w_last = (int)((unsigned)(item_end - 1) / (unsigned)run);
    return FlatSegment{item, item_end - row0 - 1, w - w_first, w_last - w_first + 1, b - row0, e - row0, w_first + item};
}

// Rows of one wave sub-tile: 16 (two MFMA row sets), i.e. 16 KiB of K and V
// at head_dim 128, whatever the number of q heads per KV head.
__host__ __device__ constexpr int subtile_rows(int hd, int g) { return (void)hd, (void)g, 16; }

// Positions one workgroup pass covers with NW waves; chunk sizes are
// multiples of it.
__host__ __device__ constexpr int rows_per_pass(int hd, int g, int nw) { return nw * subtile_rows(hd, g); }

struct StepArgs {
    const float *q;      // [n_seq][n_heads*HD], pre-RoPE
    const float *k_new;  // [n_seq][kv_dim], pre-RoPE
    const float *v_new;  // [n_seq][kv_dim]
    float *out;          // [n_seq][n_heads*HD]
    float *k_cache;      // slab base of sequence 0 at this layer
    float *v_cache;
    const float4 *rope;  // [seq_len][HD/4] of (cos_2i, sin_2i, cos_2i+1, sin_2i+1)
    const int *pos_dev;  // per-sequence positions, or nullptr -> pos_scalar
    float *ws_o;         // [n_seq][n_heads][records_per_head(grid_chunks)][HD] partial
                         // outputs: chunk records, then first-level merge records
    float2 *ws_ml;       // [n_seq][n_heads][records_per_head(grid_chunks)] (max, sum), log2 units
    int *counters;       // [n_seq][n_kv_heads][counters_per_group(grid_chunks)] arrival
                         // counters (final, then one per sub-group, kCtrStride apart),
                         // zero between launches
    long long seq_stride;// floats between sequence slabs
    int pos_scalar;
    int max_pos;         // launch was sized for positions <= max_pos
    int seq_len;
    int n_heads;
    int n_kv_heads;      // KV groups per sequence (with kv_split, twice the cache's KV heads)
    int chunk;           // positions per workgroup, a multiple of 8 (passes past its end are masked)
    int grid_chunks;     // chunks per sequence in the launch grid
    int n_groups;        // n_seq * n_kv_heads
    float scale_log2;    // log2(e) / sqrt(HD)
    int merge_asym;      // bit 0: every CU runs two workgroups of the launch, and the
                         // first-dispatched half of a group's chunks finishes first;
                         // bits 1-2: the fold helper (0 off, 1 on, 2 gives up at once)
    int spread_log2;     // a group's chunks are cut into 2^spread_log2 parts on as many
                         // XCDs (launches of fewer groups than XCDs); 0: one part
    int even_chunks;     // > 0: a sequence of T positions is cut instead into min(even_chunks, T)
                         // chunks of near-equal length (seq_chunks, chunk_start); in the
                         // slot before the 8-byte aligned pointers, so that the fields the
                         // prologue reads first keep their offsets
    float *ws_po;        // [n_groups << spread_log2][G][HD] each part's unnormalised output
    float2 *ws_pml;      // [n_groups << spread_log2][G] its (max, sum), log2 units
    FastDiv by_grid_chunks, by_kv_heads, by_chunk, by_even;  // divisions by grid_chunks, n_kv_heads,
                                                              // chunk and even_chunks (1 if 0)
    int kv_split;        // 1: n_kv_heads counts each of the cache's n_kv_heads / 2 heads twice, as
                         // two groups of G q heads (kv_group); 0: one group per head
#ifdef LEAP_TIMELINE
    unsigned long long *tl;  // this launch's [kTlMaxWgs][kTlPoints] stamps (timeline build only)
#endif
};

// The decode kernel's (and its floor kernels') leading arguments: 14 words
// that the dispatch preloads into scalar registers (the library is built
// with -mllvm -amdgpu-kernarg-preload-count=14; the code object carries a
// fallback that loads them itself where the firmware does not preload).
// They hold everything the prologue needs up to the first tile's loads
// when a launch serves one sequence at a host position, so that those
// loads do not wait for a load of the argument block (about 0.25 us on an
// idle chip); the argument block (StepArgs) follows in the kernel
// arguments and is read after they are issued.  Launches of several
// sequences or with positions on the device set w1 = kPreGeneral and read
// their prologue from the argument block.
struct Preload {
    const float *q;      // StepArgs::q
    const float *k_new;  // StepArgs::k_new
    float *k_cache;      // StepArgs::k_cache
    float *v_cache;      // StepArgs::v_cache
    const float4 *rope;  // StepArgs::rope
    uint32_t m_gc;       // StepArgs::by_grid_chunks.m
    uint32_t w0;         // grid_chunks | by_grid_chunks.s << 10 | spread_log2 << 14 | n_kv_heads << 16
    uint32_t w1;         // one sequence at a host position: pos | n_chunks << 21; else kPreGeneral
    uint32_t w2;         // the chunks: chunk c starts at min(c q + min(c, r), T), w2 = q | r << 21
};
constexpr uint32_t kPreGeneral = 0xFFFFFFFFu;
// The kernels take the words as leading scalar parameters (only those are
// preloaded), in Preload's order, ahead of the argument block.
#define LEAP_PRELOAD_PARAMS                                                                                  \
    const float *pre_q, const float *pre_k_new, float *pre_k_cache, float *pre_v_cache,                      \
        const float4 *pre_rope, uint32_t pre_m_gc, uint32_t pre_w0, uint32_t pre_w1, uint32_t pre_w2
#define LEAP_PRELOAD                                                                                         \
    Preload { pre_q, pre_k_new, pre_k_cache, pre_v_cache, pre_rope, pre_m_gc, pre_w0, pre_w1, pre_w2 }
constexpr uint32_t kPreLimit = 1u << 21;  // pos, q < kPreLimit and n_chunks, r < 2^11 for the packed words
// StepArgs' byte offset in the kernel arguments, after the preloaded words
constexpr unsigned kArgsOffset = 5 * sizeof(void *) + 4 * sizeof(uint32_t);
static_assert(kArgsOffset == 56 && alignof(StepArgs) <= 8, "argument layout");

// A kernel's argument block read at this point through a copy of the
// kernel-argument pointer that the compiler cannot see through, so that none
// of its loads (or a wait for one) is placed ahead of the loads before this
// point; offset: the block's byte offset in the kernel arguments, after the
// kernel's preloaded scalar arguments.
template <class T>
__device__ __forceinline__ T late_args(const T &host_side, unsigned offset)
{
#ifdef __HIP_DEVICE_COMPILE__
    (void)host_side;
    auto kargs = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(kargs));
    typedef __attribute__((address_space(4))) const T KernargT;
    typedef __attribute__((address_space(4))) const char KernargBytes;
    return *(KernargT *)((KernargBytes *)kargs + offset);
#else
    (void)offset;
    return host_side;
#endif
}

// The preloaded words of a launch (host side): the launch constants, and
// the positions' words when it serves one sequence at host position pos
// (one_seq), with chunk rows `chunk`, or even_chunks near-equal chunks.
inline Preload make_preload(const StepArgs &a, bool one_seq)
{
    Preload p{a.q, a.k_new, a.k_cache, a.v_cache, a.rope, a.by_grid_chunks.m, 0u, kPreGeneral, 0u};
    p.w0 = (uint32_t)a.grid_chunks | (a.by_grid_chunks.s << 10) | ((uint32_t)a.spread_log2 << 14) |
           ((uint32_t)a.n_kv_heads << 16);
    const int T = a.pos_scalar + 1;
    if (!one_seq || a.pos_dev || a.pos_scalar < 0 || a.pos_scalar >= a.seq_len || a.pos_scalar > a.max_pos ||
        (uint32_t)a.pos_scalar >= kPreLimit)
        return p;  // the kernel checks the position (and writes NaN rows for one it cannot serve)
    const int n_chunks = a.even_chunks > 0 ? (T < a.even_chunks ? T : a.even_chunks) : (T + a.chunk - 1) / a.chunk;
    const int q = a.even_chunks > 0 ? T / n_chunks : a.chunk;
    const int r = a.even_chunks > 0 ? T % n_chunks : 0;
    if ((uint32_t)q >= kPreLimit || n_chunks >= 2048) return p;
    p.w1 = (uint32_t)a.pos_scalar | ((uint32_t)n_chunks << 21);
    p.w2 = (uint32_t)q | ((uint32_t)r << 21);
    return p;
}

// ---- timeline (measurement build only) --------------------------------------
//
// Built with -DLEAP_TIMELINE (`python -m leap_amd.build` builds that library
// too, as libleap_hip_attention_tl.so), the decode kernel records
// s_memrealtime, a 100 MHz device clock, at the points below, per workgroup:
// wave 0 keeps the stamps in scalar registers, so that they add no waits, and
// stores them with the workgroup's role, XCC and hardware id when it leaves
// the kernel.  Without the define the Timeline type is empty and its marks
// compile to nothing: the production kernels are the same code.
constexpr int kTlPoints = 16;    // words per workgroup
constexpr int kTlSlots = 64;     // launches the host's ring holds
constexpr int kTlMaxWgs = 2048;  // workgroups recorded per launch
enum TlPoint {
    kTlStart = 0,      // kernel entry
    kTlPrologue,       // q rotated and shared (the prologue's barrier)
    kTlScored,         // wave 0: the first pass's scores
    kTlLoopEnd,        // wave 0: the last pass's weighted V
    kTlCombined,       // every wave's partials in LDS (the combine's barrier)
    kTlStored,         // the output or the chunk record stored
    kTlDrained,        // merge: this workgroup's record stores drained (its barrier)
    kTlCounted,        // merge: its arrival counter returned
    kTlFoldIssued,     // a fold's loads issued
    kTlFoldLoaded,     // a fold's (max, sum) pairs shared (its barrier)
    kTlFolded,         // a fold's result stored
    kTlSubCounted,     // asymmetric merge, first half: the sub-group counter returned
    kTlSubFolded,      // asymmetric merge, first half: the sub-group record stored
    kTlEnd,            // kernel exit
    kTlRole,           // role bits (kTlRole*) | arrival count << 8
    kTlHw,             // XCC id << 32 | HW_ID
};
constexpr unsigned kTlRoleSingle = 1;   // one chunk: wrote the output itself
constexpr unsigned kTlRoleFinal = 2;    // folded (part of) the final result
constexpr unsigned kTlRoleHelper = 4;   // the fold helper (second-to-last arrival)
constexpr unsigned kTlRoleSub = 8;      // folded a first-level sub-group
struct Timeline {
#ifdef LEAP_TIMELINE
    unsigned long long t[kTlPoints] = {};
    // (scheduling barriers keep the stamp in program order; a wave issues in order)
    __device__ __forceinline__ void mark(int k)
    {
        __builtin_amdgcn_sched_barrier(0);
        t[k] = __builtin_amdgcn_s_memrealtime();
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void role(unsigned r, int count)
    {
        t[kTlRole] |= r | ((unsigned long long)(unsigned)count << 8);
    }
    __device__ __forceinline__ void flush(unsigned long long *dst)
    {
        unsigned hw, xcc;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hw));
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
        t[kTlHw] = ((unsigned long long)(xcc & 0xFu) << 32) | hw;
        if (dst && threadIdx.x == 0 && blockIdx.x < (unsigned)kTlMaxWgs) {
#pragma unroll
            for (int k = 0; k < kTlPoints; k++) dst[(size_t)blockIdx.x * kTlPoints + k] = t[k];
        }
    }
#else
    __device__ __forceinline__ void mark(int) {}
    __device__ __forceinline__ void role(unsigned, int) {}
#endif
};

// The cache's KV head and the first q head of a launch's KV group kvv (of
// n_kv_heads).  With kv_split = k (1 or 2), the cache holds n_kv =
// n_kv_heads >> k heads of 2^k G q heads each, served as 2^k groups of G:
// part p is groups [p n_kv, (p + 1) n_kv), so that with n_kv a multiple of 8
// every part of a head runs on one XCD and the later reads of its rows can
// hit in L2.
struct KvGroup {
    int kvh, half, qh0;  // half: the part (0 appends the new token)
};
template <int G>
__device__ __forceinline__ KvGroup kv_group(int kvv, int n_kv_heads, int kv_split)
{
    const int n_kv = n_kv_heads >> kv_split;
    const int part = (kvv >= n_kv ? 1 : 0) + (kvv >= 2 * n_kv ? 1 : 0) + (kvv >= 3 * n_kv ? 1 : 0);
    const int kvh = kvv - part * n_kv;
    return KvGroup{kvh, part, ((kvh << kv_split) + part) * G};
}

// Whether a launch runs the PART instance of the decode kernel (the host's
// choice, restated for the floor kernels, which have no such instance):
// near-equal chunks, chunks that are not whole passes, or chunks of 2-8
// passes.
__host__ __device__ constexpr bool part_launch(int even_chunks, int chunk, int pass)
{
    return even_chunks > 0 || chunk % pass != 0 || (chunk >= 2 * pass && chunk <= 8 * pass);
}

// Chunks of a sequence of T positions, and where chunk c starts: fixed-size
// chunks of a.chunk rows (the last one shorter), or min(even_chunks, T)
// chunks of near-equal length, the first T mod n of them one row longer
// (one 32-bit quotient per sequence, ahead of the first loads).
__device__ __forceinline__ int seq_chunks(const StepArgs &a, int T)
{
    return a.even_chunks > 0 ? min(a.even_chunks, T) : (int)fast_div((uint32_t)(T + a.chunk - 1), a.by_chunk);
}
__device__ __forceinline__ int chunk_start(const StepArgs &a, int T, int n_chunks, int c)
{
    if (a.even_chunks > 0) {
        // n_chunks = min(even_chunks, T): T / even_chunks, or 1 when T < even_chunks
        const unsigned q = T >= a.even_chunks ? fast_div((uint32_t)T, a.by_even) : 1u;
        const unsigned r = (unsigned)T - q * (unsigned)n_chunks;
        return (int)((unsigned)c * q + min((unsigned)c, r));
    }
    return min(c * a.chunk, T);
}


// ---- buffer access ------------------------------------------------------------
//
// Raw buffer loads take 32-bit byte offsets from a base and return zero past
// num_records bytes, which masks rows beyond the valid range without
// branches.

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr int kRsrcWord3 = 0x00020000;  // raw 32-bit dword access, gfx9 family

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, kRsrcWord3);
}

// The loaded vector is reinterpreted whole (f32x4), never lane by lane: the
// compiler narrows a b128 buffer load to one dword when its lanes are
// bit-cast one at a time.
template <int AUX = 0>
__device__ __forceinline__ float4 buf_load4(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, AUX));
    return make_float4(v.x, v.y, v.z, v.w);
}

template <int AUX = 0>
__device__ __forceinline__ float2 buf_load2(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    const f32x2 v = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, AUX));
    return make_float2(v.x, v.y);
}

template <int AUX = 0>
__device__ __forceinline__ void buf_store4(__amdgpu_buffer_rsrc_t r, uint32_t off, float4 x)
{
    const f32x4 v = {x.x, x.y, x.z, x.w};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, (int)off, 0, AUX);
}

template <int AUX = 0>
__device__ __forceinline__ void buf_store2(__amdgpu_buffer_rsrc_t r, uint32_t off, float2 x)
{
    const f32x2 v = {x.x, x.y};
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, (int)off, 0, AUX);
}

// ---- wave helpers ---------------------------------------------------------
//
// The q.K scores come out of 4x4x1 MFMAs with lane = 32*kq + 4*ksl + kj
// holding the partial dot product of K row 4*kq + kj of an 8-row set over dim
// slice ksl (eight slices).  The slices are summed with DPP inside each 16-lane
// row (row_ror by 4 and by 8 lanes add the lanes of equal kj) and then across
// the row pair, for the sub-tile's two 8-row sets at once: v_permlane16_swap
// hands the odd rows of the first set's register and the even rows of the
// second's to each other, and one addition leaves the first set's scores in
// rows 0 and 2 and the second's in rows 1 and 3 (slice_sum2).  One register
// then holds the 16 rows of the sub-tile (score_row: the lane's row), each in
// four lanes, and the softmax works on half the registers that one set each
// would take.  The wave max / sum takes the quad (kj) with DPP and the four
// rows with v_readlane, which leaves a wave-uniform result.

template <int CTRL>
__device__ __forceinline__ float dpp(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL,
                                                              0xF, 0xF, true));
}

__device__ __forceinline__ float lane_value(float x, int lane)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}

// Sums of the eight dim slices of two row sets' scores: x's in the even
// 16-lane rows, y's in the odd ones.
__device__ __forceinline__ float slice_sum2(float x, float y)
{
    x += dpp<0x124>(x);  // row_ror:4
    y += dpp<0x124>(y);
    x += dpp<0x128>(x);  // row_ror:8
    y += dpp<0x128>(y);
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, y),
                                                    false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
// The sub-tile row whose score slice_sum2 leaves in a lane.
__device__ __forceinline__ int score_row(int lane) { return 8 * ((lane >> 4) & 1) + 4 * (lane >> 5) + (lane & 3); }

// Max / sum over R rows of 16 lanes (R = 1, 2 or 4): rows 2k and 2k + 1
// meet, then the two halves of the wave, through the lane crossbar
// (ds_bpermute: no LDS storage, no barrier).  Every lane ends with the
// result of its rows, the same bits in each (a + b == b + a).  The
// permlane swaps would be cheaper, but given one value as both operands the
// compiler takes their two results for one and folds max(p0, p1) to p0 and
// p0 + p1 to p0 + p0.
template <int R, bool MAX>
__device__ __forceinline__ float rows_reduce(float x)
{
    auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
    if constexpr (R >= 2) x = op(x, __shfl_xor(x, 16));
    if constexpr (R >= 4) x = op(x, __shfl_xor(x, 32));
    return x;
}

// Max / sum over a sub-tile's rows of a value that is uniform across the four
// lanes of each row; wave-uniform result.
__device__ __forceinline__ float score_rows_max(float x)
{
    x = fmaxf(x, dpp<0xB1>(x));  // quad_perm [1,0,3,2]
    x = fmaxf(x, dpp<0x4E>(x));  // quad_perm [2,3,0,1]
    return fmaxf(fmaxf(lane_value(x, 0), lane_value(x, 16)), fmaxf(lane_value(x, 32), lane_value(x, 48)));
}

__device__ __forceinline__ float score_rows_sum(float x)
{
    x += dpp<0xB1>(x);
    x += dpp<0x4E>(x);
    return (lane_value(x, 0) + lane_value(x, 16)) + (lane_value(x, 32) + lane_value(x, 48));
}

// acc += a[c] * b[c] for the four float4 components, one 4x4x1 MFMA each:
// block k = lane / 4 adds A_k (4x1, lane 4k+i gives row i) times B_k (1x4,
// lane 4k+j gives column j) to its 4x4 tile, held as column j in lane 4k+j.
__device__ __forceinline__ f32x4 mfma4(float4 a, float4 b, f32x4 acc)
{
    acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a.x, b.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a.y, b.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a.z, b.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a.w, b.w, acc, 0, 0, 0);
    return acc;
}

__device__ __forceinline__ void fma4(float4 &acc, float p, float4 v)
{
    acc.x += p * v.x;
    acc.y += p * v.y;
    acc.z += p * v.z;
    acc.w += p * v.w;
}

__device__ __forceinline__ void scale4(float4 &acc, float s)
{
    acc.x *= s;
    acc.y *= s;
    acc.z *= s;
    acc.w *= s;
}

// Lane src's float4 (every lane of the wave active).
__device__ __forceinline__ float4 lane_float4(float4 v, int src)
{
    const int b = src * 4;
    return make_float4(__int_as_float(__builtin_amdgcn_ds_bpermute(b, __float_as_int(v.x))),
                       __int_as_float(__builtin_amdgcn_ds_bpermute(b, __float_as_int(v.y))),
                       __int_as_float(__builtin_amdgcn_ds_bpermute(b, __float_as_int(v.z))),
                       __int_as_float(__builtin_amdgcn_ds_bpermute(b, __float_as_int(v.w))));
}

// Interleaved-pair rotation of one float4 (two pairs) with table entry
// t = (cos_a, sin_a, cos_b, sin_b), products rounded separately as the
// reference's mul/mul/addsub body does (FloatTransformer.cpp:461-464).
__device__ __forceinline__ float4 rope4(float4 x, float4 t)
{
#pragma clang fp contract(off)
    float4 r;
    r.x = x.x * t.x - x.y * t.y;
    r.y = x.y * t.x + x.x * t.y;
    r.z = x.z * t.z - x.w * t.w;
    r.w = x.w * t.z + x.z * t.w;
    return r;
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// One register of two: the lower half of the lanes gets the sum of x's two
// halves, the upper half the sum of y's.
__device__ __forceinline__ float halves_sum2(float x, float y)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, y),
                                                    false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
// The same within each pair of 16-lane rows.
__device__ __forceinline__ float rows_sum2(float x, float y)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, y),
                                                    false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}

// ---- the fused decode-attention kernel --------------------------------------

// Growth of the running max (log2 units) tolerated before the accumulators
// are rescaled: p = 2^(s - m_ref) stays below 2^kLazyMax.
constexpr float kLazyMax = 8.0f;
// The reference max before any score: the lowest finite value.
constexpr float kLowest = -3.402823466e+38f;

template <int HD, int G, int NW>
struct Shape {
    static constexpr int THREADS = NW * kWave;
    static constexpr int GQ = (G + 3) / 4;                 // head quads (MFMA tile rows)
    static constexpr int NF = HD / 32;                     // K float4 per lane per row set
    static constexpr int R = subtile_rows(HD, G);          // rows per wave sub-tile
    static constexpr int KS = R / 8;                       // K row sets (8 rows) per sub-tile
    static constexpr int LPV = HD / 4;                     // lanes per V row
    static constexpr int RPV = kWave / LPV;                // V rows per load set
    static constexpr int VS = R / RPV;                     // V load sets per sub-tile
    static constexpr int ROWS = NW * R;                    // positions per workgroup pass
    static constexpr int D4 = HD / 4;                      // float4 per head row
    // merge: heads padded to a power of two (3 -> 4), chunk lanes per head
    static constexpr int GM = G <= 1 ? 1 : G <= 2 ? 2 : G <= 4 ? 4 : 8;
    static constexpr int MG = THREADS / (GM * D4);
    static_assert(HD % 32 == 0, "head_dim vs K slices");
    static_assert(KS == 2 && R % RPV == 0, "sub-tile shape");
    static_assert(G <= 8, "q heads per KV head");
    static_assert(MG >= 1 && THREADS % (GM * D4) == 0, "merge layout");
};

// The sums of a wave's output accumulators over its V row slots (lanes of
// equal dims: the halves of the wave at head_dim 128, its four 16-lane rows at
// 64), put(first, head, dims 4*vj .. +3) in one lane per (head, column); first
// is the lowest head of that register, a constant once unrolled.  The swaps
// that bring two registers' slots together leave one head per half (row), so
// that a quad of heads takes two (one) 16-byte writes per lane to LDS in place
// of four, and the waves' combine reads half (a quarter) of the bytes.
template <int HD, int G, class Put>
__device__ __forceinline__ void slot_sums(const f32x4 (&acc)[(G + 3) / 4][4], int lane, Put put)
{
#pragma unroll
    for (int q = 0; q < (G + 3) / 4; q++) {
        // head 4q + i's component e; zero past the heads
        auto at = [&](int i, int e) { return 4 * q + i < G ? acc[q][e][i] : 0.0f; };
        if constexpr (HD == 128) {
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                if (4 * q + i >= G) continue;
                const int h = 4 * q + i + (lane >> 5);
                const float4 o = make_float4(halves_sum2(at(i, 0), at(i + 1, 0)), halves_sum2(at(i, 1), at(i + 1, 1)),
                                             halves_sum2(at(i, 2), at(i + 1, 2)), halves_sum2(at(i, 3), at(i + 1, 3)));
                if (h < G) put(4 * q + i, h, o);
            }
        } else {
            // rows 0-3 of the wave: heads 0, 1, 2, 3 of the quad
            const int h = 4 * q + (lane >> 4);
            float c[4];
#pragma unroll
            for (int e = 0; e < 4; e++)
                c[e] = halves_sum2(rows_sum2(at(0, e), at(1, e)), rows_sum2(at(2, e), at(3, e)));
            if (h < G) put(4 * q, h, make_float4(c[0], c[1], c[2], c[3]));
        }
    }
}

// MFMA: the score and weighted-V products on the matrix cores (4x4x1 f32
// MFMAs); false: the same products as per-lane VALU FMAs, leaving the same
// partial sums in the same lanes (the A/B of the matrix-core choice).
// PART: chunks that need not be whole passes (near-equal chunks, or forced
// sizes that are multiples of 8): rows past a chunk's end are masked, only
// the chunk holding pos writes the new token, and a chunk's passes start at
// pass chunk_id mod n_sub.  The host also runs it for chunks of 2-8 whole
// passes, for that rotation.  One-pass and long-run launches use PART =
// false, whose prologue is shorter (the two measured 0.07-0.14 us apart per
// launch at Llama-3-8B ctx 4096 and TinyLlama ctx 256).
// The wait of the second-to-last arrival of a one-level fold that shares
// the fold with the last arrival (one thread): poll the final counter, at
// most kHelpPolls times (none in mode 2, which tests the fallback), until
// the last arrival has counted in.  Returns 1 if this workgroup folds its
// half of the heads, and then resets the counter.  On giving up it adds
// kGiveUp to the counter: if the last arrival has counted in meanwhile
// (the add returns target), it folds its half of the heads only and this
// workgroup still folds the other half; otherwise the last arrival sees
// kGiveUp, folds every head and resets the counter, and this returns 0.
// Every head is folded once and the counter reset once, in any order.
__device__ __forceinline__ int fold_helper_wait(int *ctr, int target, int mode)
{
    const int polls = mode == 2 ? 0 : kHelpPolls;
    for (int i = 0; i < polls; i++) {
        if (__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == target) {
            *ctr = 0;
            return 1;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    if (__hip_atomic_fetch_add(ctr, kGiveUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == target) {
        *ctr = 0;
        return 1;
    }
    return 0;
}

// The new token's cache rows, when the decode body leaves their stores to
// the kernel's end: the rotated k and v_new of float4 column L in lane L.
struct NewRow {
    float4 k, v;
    float *kdst, *vdst;
    bool on;
};

// FLAT: the body serves one segment of a flat launch, fs; a workgroup runs it
// once per segment.
template <int HD, int G, int NW, bool MFMA, bool PART, int KVS, bool FLAT = false>
__device__ __forceinline__ void decode_attention_body(const StepArgs &args, const Preload &pre, Timeline &tl,
                                                      NewRow &nr, const FlatSegment &fs = FlatSegment{})
{
    using S = Shape<HD, G, NW>;
    constexpr int GQ = S::GQ, NF = S::NF, R = S::R, KS = S::KS;
    constexpr int LPV = S::LPV, RPV = S::RPV, VS = S::VS, D4 = S::D4, GM = S::GM, MG = S::MG;
    // Where the new token's row (position pos) joins the scores and the
    // weighted V.  Up to 4 q heads per KV head: after the loop, by the wave
    // whose rows hold pos, with a score of its own (a dot product per head
    // and a lane reduction); the loop masks row pos like the rows past it.
    // Keeping the row out of the loop's products frees 60-100 registers of
    // the loop (Llama-3-8B heads: 191 -> 120 VGPRs in the 4-wave partial-
    // pass instance, 222 -> 123 in the whole-pass one, 190 -> 130 on 2
    // waves), which measured faster with
    // graph replay at every context of those heads: ctx 8192 15.50 -> 14.10
    // us, 16384 25.59 -> 25.00, 2304 8.34 -> 8.16, 4096 9.63 -> 9.54.  With 8
    // q heads the row stays in the loop's products (staged into the K and V
    // registers of the row's load): added afterwards it measured slower for
    // them (TinyLlama ctx 256 5.55 -> 6.18 us, Llama-3-405B ctx 4096 15.75 ->
    // 17.06), eight heads of dependent reductions in one wave.
    constexpr bool NEW_AFTER = G <= 4;

    // id = ((pg / 8) * grid_chunks + lc) * 8 + pg % 8, where the part-group
    // pg = group * 2^spread_log2 + part covers the group's chunks
    // [part * grid_chunks, (part + 1) * grid_chunks) and lc is the chunk
    // within the part.  Every workgroup of a part-group runs on one XCD.
    const int xcd = blockIdx.x % kXcds;
    const int local = blockIdx.x / kXcds;
    const int grid_chunks = (int)(pre.w0 & 1023u);
    const int spread_log2 = (int)((pre.w0 >> 14) & 3u);
    const int n_kv_heads = (int)(pre.w0 >> 16);
    const int lq = (int)fast_div((uint32_t)local, FastDiv{pre.m_gc, (pre.w0 >> 10) & 15u});
    const int lc = FLAT ? fs.lc : local - lq * grid_chunks;
    const int pgroup = (FLAT ? fs.item : lq) * kXcds + xcd;
    const int group = FLAT ? pgroup : pgroup >> spread_log2;
    const int part = FLAT ? 0 : pgroup & ((1 << spread_log2) - 1);
    const int chunk_id = FLAT ? lc : part * grid_chunks + lc;  // within the group
    // The sequence, its position, its chunks (chunk c starts at
    // min(c cq + min(c, cr), T)) and its slab: from the preloaded words for
    // one sequence at a host position, else from the argument block, whose
    // fields are loaded as one batch before the first branch there (an
    // empty asm that takes them as inputs): left to the compiler, each load
    // follows the branch that first needs it, one dependent round trip
    // after another.
    int seq, pos, n_chunks, cq, cr;
    size_t slab;
    if constexpr (FLAT) {
        seq = (int)fast_div((uint32_t)group, args.by_kv_heads);
        pos = fs.pos;
        n_chunks = fs.n_local;
        cq = cr = 0;
        slab = (size_t)seq * (size_t)args.seq_stride;
    } else if (pre.w1 != kPreGeneral) {
        if (group >= n_kv_heads) return;
        seq = 0;
        pos = (int)(pre.w1 & (kPreLimit - 1));
        n_chunks = (int)(pre.w1 >> 21);
        cq = (int)(pre.w2 & (kPreLimit - 1));
        cr = (int)(pre.w2 >> 21);
        slab = 0;
    } else {
        asm volatile("" ::"s"(args.pos_dev), "s"(args.seq_stride), "s"(args.pos_scalar), "s"(args.max_pos),
                     "s"(args.seq_len), "s"(args.n_heads), "s"(args.chunk), "s"(args.n_groups),
                     "s"(args.even_chunks), "s"(args.by_kv_heads.m), "s"(args.by_kv_heads.s), "s"(args.by_chunk.m),
                     "s"(args.by_chunk.s), "s"(args.by_even.m), "s"(args.by_even.s), "s"(args.out));
        if (pgroup >= (args.n_groups << spread_log2)) return;
        seq = (int)fast_div((uint32_t)group, args.by_kv_heads);
        pos = args.pos_dev ? args.pos_dev[seq] : args.pos_scalar;
        if (pos < 0 || pos >= args.seq_len || pos > args.max_pos) {
            // A device position the launch cannot serve: no row is read or
            // written, and the sequence's output rows read NaN so that the
            // skip is visible (the first chunk of each group writes its
            // heads; a spread launch's merge launch does it instead).
            const int kvv = group - seq * n_kv_heads;
            const int qh0 = KVS ? kv_group<G>(kvv, n_kv_heads, KVS).qh0 : kvv * G;
            if (chunk_id == 0 && spread_log2 == 0)
                for (int i = threadIdx.x; i < G * HD; i += NW * kWave)
                    args.out[(size_t)seq * args.n_heads * HD + (size_t)qh0 * HD + i] = __builtin_nanf("");
            return;
        }
        const int T = pos + 1;
        n_chunks = PART ? seq_chunks(args, T) : (int)fast_div((uint32_t)(T + args.chunk - 1), args.by_chunk);
        if (args.even_chunks > 0) {
            // n_chunks = min(even_chunks, T): T / even_chunks, or 1 when T < even_chunks
            cq = T >= args.even_chunks ? (int)fast_div((uint32_t)T, args.by_even) : 1;
            cr = T - cq * n_chunks;
        } else {
            cq = args.chunk;
            cr = 0;
        }
        slab = (size_t)seq * (size_t)args.seq_stride;
    }
    const int kvv = group - seq * n_kv_heads;  // the group within its sequence
    // KVS: 2^KVS launch groups per cache head (kv_split = KVS), compiled as
    // instances of their own so that the others keep their code
    const KvGroup kg = KVS ? kv_group<G>(kvv, n_kv_heads, KVS) : KvGroup{kvv, 0, kvv * G};
    const int kvh = kg.kvh;
    const bool store_new = kg.half == 0;  // the one group per cache head that appends the new token
    int tid = threadIdx.x;
    // (what follows from the thread's number is worked out again for each
    // segment: held through the ones before, it took 256 registers and scratch)
    if constexpr (FLAT) asm volatile("" : "+v"(tid));
    // (scalar with PART, whose tests of the wave's rows it makes scalar too; in
    // the whole-pass instances it measured 0.5-1% slower at ctx 2048-4096)
    const int wave = PART ? __builtin_amdgcn_readfirstlane(tid / kWave) : tid / kWave;
    const int lane = tid % kWave;

    const int T = pos + 1;
    if (chunk_id >= n_chunks) return;
    // chunks of this part (at least 1 here)
    const int n_local = FLAT ? n_chunks : min(grid_chunks, n_chunks - part * grid_chunks);

    const int kv_dim = (n_kv_heads >> KVS) * HD;
    const int q_dim = n_kv_heads * G * HD;  // every q head of a sequence
    const uint32_t row_bytes = (uint32_t)kv_dim * 4u;
    float *kc = pre.k_cache + slab + (size_t)kvh * HD;
    float *vc = pre.v_cache + slab + (size_t)kvh * HD;
    // This chunk's rows [chunk_begin, last].  With PART a pass may reach past
    // the chunk's end.  Rows up to min(pos, chunk end) of this KV head are in
    // range: row pos (the new token, from registers) and the rows beyond
    // read 0 without touching memory, and their scores are masked (row pos
    // too when it is added after the loop).
    constexpr int LAST_NEW = NEW_AFTER ? 1 : 0;
    int chunk_begin, chunk_end, row_end, last;
    if constexpr (PART) {
        chunk_begin = FLAT ? fs.begin : min(chunk_id * cq + min(chunk_id, cr), T);
        chunk_end = FLAT ? fs.end : min((chunk_id + 1) * cq + min(chunk_id + 1, cr), T);
        row_end = min(pos, chunk_end);
        last = min(pos - LAST_NEW, chunk_end - 1);
    } else {
        chunk_begin = chunk_id * cq;
        chunk_end = min(chunk_begin + cq, T);
        row_end = pos;
        last = pos - LAST_NEW;
    }
    const __amdgpu_buffer_rsrc_t k_rsrc = make_rsrc(kc, (uint32_t)row_end * row_bytes);
    const __amdgpu_buffer_rsrc_t v_rsrc = make_rsrc(vc, (uint32_t)row_end * row_bytes);
    const float *k_row_new = pre.k_new + (size_t)seq * kv_dim + (size_t)kvh * HD;
    const float *qg = pre.q + (size_t)seq * q_dim + (size_t)kg.qh0 * HD;
    const float4 *rope_row = pre.rope + (size_t)pos * (HD / 4);

    __shared__ __align__(16) float p_lds[NW][R * G];
    __shared__ float4 q_lds[G][HD / 4];  // rotated, scaled q of the group's heads
    // The waves' partial outputs, [wave][V row slot][head][column]; also staging
    // for the new token (per wave) and the merge's scratch.  With PART a wave
    // sums its slots first (slot_sums), which in flat launches also halves (or
    // quarters) the bytes of every flush.  With the probabilities read ahead
    // (below), same process, back to back: Llama-3-8B heads ctx 256 5.07 ->
    // 4.93 us, ctx 1000 5.84 -> 5.66, TinyLlama ctx 256 within 2%, ctx 1000
    // 5.43 -> 5.25, Llama-3.1-405B ctx 4096 14.5 -> 14.1.  Whole-pass launches
    // keep the slots apart: the same steps made Llama-3-8B ctx 4096 0.8%
    // slower.
    constexpr int SLOTS = PART ? 1 : RPV;
    // (a float4 per lane and wave at least, for the staging and the merge)
    constexpr int CSLOTS = SLOTS * G * D4 < kWave ? (kWave + G * D4 - 1) / (G * D4) : SLOTS;
    __shared__ float4 comb_o[NW][CSLOTS][G][D4];
    __shared__ __align__(16) float comb_l[G][NW];  // [head][wave]: a head's NW values in one read
    __shared__ __align__(16) float comb_m[G][NW];
    // FLAT: the new token's staging, apart from the combine buffer, which holds
    // the waves' flushed sums during the loop
    __shared__ float4 stage_lds[FLAT ? NW : 1][FLAT ? 2 * D4 : 1];
    __shared__ float2 ml_lds[GM * kFinalMax];  // the asymmetric merge's final (max, sum) pairs
    __shared__ int s_last;

    // K layout, for the score MFMAs: lane = 32*kq + 4*ksl + kj holds row
    // krow = 4*kq + kj of each 8-row set, dims 32*f + 4*ksl .. +3 for
    // f < HD/32, so one load instruction reads 128 contiguous bytes of each of
    // eight rows.  MFMA block lane/4 = 8*kq + ksl multiplies four q heads
    // (A: lane 4*block + i gives head 4*quad + i) by its four rows (B) at one
    // dim; the eight slices are summed afterwards (slice_sum2).
    const int kj = lane & 3, ksl = (lane >> 2) & 7, kq = lane >> 5;
    const int krow = 4 * kq + kj;
    const int srow = score_row(lane);  // the row whose score this lane holds
    // V layout: lane = vg*LPV + vj; lane holds dims 4*vj .. +3.
    const int vg = lane / LPV, vj = lane % LPV;

    // Prologue.  The group's q heads are loaded once per workgroup (one pair
    // per thread) ahead of the first K/V tile, rotated with the score scale
    // folded in, and shared through LDS; only the workgroup whose chunk holds
    // pos loads and rotates the new token's k and v.
    // passes over this chunk's rows that reach a position <= pos
    const int n_sub = PART ? (chunk_end - chunk_begin + S::ROWS - 1) / S::ROWS
                           : (min(cq, T - chunk_begin) + S::ROWS - 1) / S::ROWS;
    const bool has_pos = (chunk_id == n_chunks - 1);
    constexpr int PAIRS = G * HD / 2;
    constexpr int QP = (PAIRS + S::THREADS - 1) / S::THREADS;  // q pairs per thread
    const float2 *rope2 = reinterpret_cast<const float2 *>(rope_row);
    float2 qp[QP], qt[QP];
#pragma unroll
    for (int i = 0; i < QP; i++) {
        const int pair = tid + i * S::THREADS;
        if (pair < PAIRS) qp[i] = reinterpret_cast<const float2 *>(qg)[pair];
        // every thread: lane L holds table pair L mod HD/2 (THREADS is a
        // multiple of HD/2), which the new token's k rotation reads too
        qt[i] = rope2[pair % (HD / 2)];
    }
    float4 kb[KS][NF], vb[VS];
    auto load_k = [&](int sub) {
        const int base = chunk_begin + (sub * NW + wave) * R;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const uint32_t roff = (uint32_t)(base + ks * 8 + krow) * row_bytes;
#pragma unroll
            for (int f = 0; f < NF; f++)
                kb[ks][f] = buf_load4<kNt>(k_rsrc, roff + 16u * (uint32_t)(8 * f + ksl));
        }
    };
    auto load_v = [&](int sub) {
        const int base = chunk_begin + (sub * NW + wave) * R;
#pragma unroll
        for (int vs = 0; vs < VS; vs++) {
            const uint32_t roff = (uint32_t)(base + vs * RPV + vg) * row_bytes;
            vb[vs] = buf_load4<kNt>(v_rsrc, roff + 16u * (uint32_t)vj);
        }
    };
    // q: rotate (fused multiply-adds are fine, q is not stored) and scale so
    // scores come out in log2 units.  The fused product of each pair is
    // spelled out, so that the rounding does not depend on which product the
    // compiler would have fused.
    float *q_flat = reinterpret_cast<float *>(&q_lds[0][0]);
    auto rotate_q = [&](float scale_log2) {
#pragma clang fp contract(off)
#pragma unroll
        for (int i = 0; i < QP; i++) {
            const int pair = tid + i * S::THREADS;
            if (pair < PAIRS) {
                const float x0 = qp[i].x, x1 = qp[i].y, c = qt[i].x, sn = qt[i].y;
                q_flat[2 * pair] = __builtin_fmaf(x0, c, -(x1 * sn)) * scale_log2;
                q_flat[2 * pair + 1] = __builtin_fmaf(x0, sn, x1 * c) * scale_log2;
            }
        }
    };

    // First tile, in the order q and its table pairs (above), the new
    // token's k, K rows, V rows, the new token's v.  Every workgroup issues
    // the new token's loads, one per wave each, through descriptors that are
    // empty outside the workgroup holding pos (those loads return 0 without
    // touching memory): without a branch, the waits (which count outstanding
    // loads in issue order) stay exact, and the prologue barrier waits for q
    // alone.  Added in the loop (8 q heads), the wave holding pos takes its
    // lanes' parts of the k row through LDS, next to the table row (the q
    // pairs' table entries), and of the v row across lanes; added after the
    // loop, lane L < HD/4 rotates and scores float4 L of the row.
    const uint32_t new_bytes = has_pos ? (uint32_t)HD * 4u : 0u;
    const __amdgpu_buffer_rsrc_t kn_rsrc = make_rsrc(k_row_new, new_bytes);
    // (scheduling barriers keep the compiler from reordering the groups)
    // With PART, passes start at pass chunk_id mod n_sub and wrap around.
    // A launch's chunks start at equal strides, and when the stride is a
    // power of two the chunks' streams otherwise sit at the same offset of
    // their rows at once (Llama-3-8B ctx 8192, 128-row chunks: 20.3 -> 17.0
    // us per launch; 64 q heads: 26.0 -> 18.5 us; ctx 16384: 30.1 -> 26.0).
    // Rotating among the full passes only, so that a partial last pass is
    // never the first (whose loads cannot be skipped), measured slower at
    // ctx 8200 and 12000 (+0.2 and +0.5 us): fewer phases among the chunks.
    const int sub0 = (PART && n_sub > 1) ? chunk_id % n_sub : 0;
    // lane L < HD/4 holds float4 L of k_new (of v_new below), the other
    // lanes read past the range, 0; k_new goes ahead of the K rows, so that
    // the wave holding pos has it staged before its rows arrive
    const float4 knew_l = buf_load4(kn_rsrc, 16u * (uint32_t)lane);
    __builtin_amdgcn_sched_barrier(0);
    load_k(sub0);
    __builtin_amdgcn_sched_barrier(0);
    load_v(sub0);
    __builtin_amdgcn_sched_barrier(0);
    // The argument block, from here on (read after the loads above).
    const StepArgs a = late_args(args, kArgsOffset);
    // every field the rest reads, as one batch of loads
    asm volatile("" ::"s"(a.v_new), "s"(a.scale_log2), "s"(a.out), "s"(a.ws_o), "s"(a.ws_ml), "s"(a.counters),
                 "s"(a.merge_asym), "s"(a.ws_po), "s"(a.ws_pml));
    const float *v_row_new = a.v_new + (size_t)seq * kv_dim + (size_t)kvh * HD;
    const __amdgpu_buffer_rsrc_t vn_rsrc = make_rsrc(v_row_new, new_bytes);
    const float4 vnew_l = buf_load4(vn_rsrc, 16u * (uint32_t)lane);
    __builtin_amdgcn_sched_barrier(0);
    rotate_q(a.scale_log2);
    // The table row, for the new token's k, in this wave's combine buffer
    // (unused until the waves combine): float4 [D4, 2*D4); the k_new row
    // goes to [0, D4) when it is needed.
    float4 *nt_lds = FLAT ? &stage_lds[FLAT ? wave : 0][0] : &comb_o[wave][0][0][0];
    static_assert(CSLOTS * G >= 2, "new-token staging");
    if (lane < HD / 2) reinterpret_cast<float2 *>(nt_lds + D4)[lane] = qt[0];
    __syncthreads();
    tl.mark(kTlPrologue);
    // Score MFMA A operand: head 4*quad + kj at this lane's dims (zero for
    // the unused heads of a partial quad).
    float4 qa[GQ][NF];
#pragma unroll
    for (int qd = 0; qd < GQ; qd++)
#pragma unroll
        for (int f = 0; f < NF; f++)
            qa[qd][f] = (4 * qd + kj < G) ? q_lds[4 * qd + kj][8 * f + ksl] : make_float4(0.f, 0.f, 0.f, 0.f);

    // P.V accumulators, MFMA 4x4x1 (16 blocks) layout: block b = lane / 4
    // covers the lanes of one V row; acc[q][e][i] is head 4q+i at dim
    // 4*vj + e of the rows this lane's half (or quarter) of the wave sees.
    float m_ref[G], l_run[G];
    f32x4 acc[GQ][4];
#pragma unroll
    for (int h = 0; h < G; h++) {
        m_ref[h] = kLowest;
        l_run[h] = 0.0f;
    }
#pragma unroll
    for (int q = 0; q < GQ; q++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[q][e] = f32x4{0.f, 0.f, 0.f, 0.f};

    // FLAT: this wave's outputs so far, relative to 2^m_sum, as its partials in
    // the combine buffer, and its sums of p
    float m_sum[FLAT ? G : 1], l_sum[FLAT ? G : 1];
    bool flushed = false;
    auto flush = [&]() {
        float ratio[G];  // from the sums' reference max to the current one
#pragma unroll
        for (int h = 0; h < G; h++) {
            ratio[h] = flushed ? fast_exp2(m_sum[h] - m_ref[h]) : 0.0f;
            m_sum[h] = m_ref[h];
            l_sum[h] = flushed ? ratio[h] * l_sum[h] + l_run[h] : l_run[h];
            l_run[h] = 0.0f;
        }
        slot_sums<HD, G>(acc, lane, [&](int h0, int h, float4 o) {
            float4 *dst = &comb_o[wave][0][h][vj];
            if (flushed) {
                auto of = [&](int j) { return ratio[h0 + j < G ? h0 + j : 0]; };
                if constexpr (HD == 128)
                    fma4(o, lane >> 5 ? of(1) : of(0), *dst);
                else
                    fma4(o, lane >> 5 ? (lane & 16 ? of(3) : of(2)) : (lane & 16 ? of(1) : of(0)), *dst);
            }
            *dst = o;
        });
        flushed = true;
    };

    for (int i = 0; i < n_sub; i++) {
        if constexpr (FLAT) {
            if (i > 0 && i % kFlatFlushPasses == 0) {
                flush();
#pragma unroll
                for (int q = 0; q < GQ; q++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[q][e] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
        const int sub = sub0 + i < n_sub ? sub0 + i : sub0 + i - n_sub;
        const int base = chunk_begin + (sub * NW + wave) * R;
        // A later pass whose rows for this wave all lie past the chunk's end
        // (the partial last pass) is skipped by the wave: no loads, nothing
        // to add.  Every load of the earlier passes has been waited for, so
        // both ways leave the same loads outstanding.
        if (PART && i > 0 && base >= chunk_end) continue;
        if (i > 0) {
            load_k(sub);
            load_v(sub);
            // Every load of the pass goes out before its products.  Below
            // 128 VGPRs the compiler's scheduler, aiming at more waves per
            // SIMD, moved each load next to its first use, into the register
            // that the previous product had just freed, which put a memory
            // round trip between products of one pass: Llama-3.1-8B ctx
            // 131072 (one workgroup per CU, 64 passes per chunk) 157 -> 188
            // us per launch.
            __builtin_amdgcn_sched_barrier(0);
        }

        // The new token's row, in the loop (8 q heads): k_new, rotated
        // exactly as the reference rotates it (it is stored), and v_new are
        // appended to
        // cache[layer][pos] and replace the (zero) loads of that row, k here
        // (the scores wait for the K loads anyway) and v just before the
        // weighted V (it is loaded last): overwriting a register whose load
        // is still in flight, or storing a loaded value, first waits for
        // that load.
        const bool pos_here = !NEW_AFTER && (!PART || has_pos) && pos >= base && pos < base + R;  // wave-uniform
        if (pos_here) {
            // k_new through the wave's staging: each lane reads its dims
            // 32*f + 4*ksl .. +3 of k_new and of the table row
            if (lane < D4) nt_lds[lane] = knew_l;
            __builtin_amdgcn_wave_barrier();
            // (one column at a time: the loop's registers are all live here)
#pragma unroll
            for (int f = 0; f < NF; f++) {
                const float4 knew = rope4(nt_lds[8 * f + ksl], nt_lds[D4 + 8 * f + ksl]);
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    const int t = base + ks * 8 + krow;
                    if (t == pos) {
                        kb[ks][f] = knew;
                        if (store_new) *reinterpret_cast<float4 *>(kc + (size_t)t * kv_dim + 4 * (8 * f + ksl)) = knew;
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        // Scores (log2 units) on the matrix cores: s[h] is head h at row srow
        // of the sub-tile, -inf past pos.
        float s[G];
        {
            const bool ok = base + srow <= last;
#pragma unroll
            for (int qd = 0; qd < GQ; qd++) {
                f32x4 d[KS];
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    d[ks] = f32x4{0.f, 0.f, 0.f, 0.f};
                    if constexpr (MFMA) {
#pragma unroll
                        for (int f = 0; f < NF; f++) d[ks] = mfma4(qa[qd][f], kb[ks][f], d[ks]);
                    } else {
                        // lane (kq, ksl, kj): head 4*qd + i times row 4*kq + kj
                        // over this lane's dims, the partial the MFMA leaves in
                        // d[i]
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            if (4 * qd + i >= G) continue;
#pragma unroll
                            for (int f = 0; f < NF; f++) {
                                const float4 qv = q_lds[4 * qd + i][8 * f + ksl];
                                d[ks][i] += qv.x * kb[ks][f].x + qv.y * kb[ks][f].y + qv.z * kb[ks][f].z + qv.w * kb[ks][f].w;
                            }
                        }
                    }
                }
                // cross-lane: every lane takes part
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (4 * qd + i >= G) continue;
                    const float v = slice_sum2(d[0][i], d[1][i]);
                    s[4 * qd + i] = ok ? v : -INFINITY;
                }
            }
        }

        // Online softmax with a lazily raised reference max: only when some
        // score exceeds m_ref + kLazyMax is the wave max taken and the
        // accumulators rescaled (always on the first tile with a valid row:
        // m_ref starts at the lowest finite value, from which any other
        // finite score is further away than kLazyMax).  A masked score is
        // -inf, and 2^(-inf - m_ref) is 0.
        float t[G], over = -INFINITY;
#pragma unroll
        for (int h = 0; h < G; h++) {
            t[h] = s[h] - m_ref[h];
            over = fmaxf(over, t[h]);
        }
        if (i == 0) tl.mark(kTlScored);
        if (__builtin_amdgcn_ballot_w64(over > kLazyMax) != 0) {
#pragma unroll
            for (int h = 0; h < G; h++) {
                const float m_new = fmaxf(m_ref[h], score_rows_max(s[h]));
                const float alpha = fast_exp2(m_ref[h] - m_new);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[h / 4][e][h % 4] *= alpha;
                l_run[h] *= alpha;
                m_ref[h] = m_new;
                t[h] = s[h] - m_new;
            }
        }
        // (the four lanes of a row hold the same p: l is kept per lane and
        // summed over the rows once at the end)
#pragma unroll
        for (int h = 0; h < G; h++) {
            s[h] = fast_exp2(t[h]);
            l_run[h] += s[h];
        }

        // Probabilities to LDS, [row][head], from one lane per row.
        if ((lane & 0xC) == 0) {
            float *dst = &p_lds[wave][srow * G];
            if constexpr (G % 4 == 0) {
#pragma unroll
                for (int qd = 0; qd < GQ; qd++)
                    reinterpret_cast<float4 *>(dst)[qd] = make_float4(s[4 * qd], s[4 * qd + 1], s[4 * qd + 2], s[4 * qd + 3]);
            } else {
#pragma unroll
                for (int h = 0; h < G; h++) dst[h] = s[h];
            }
        }
        __builtin_amdgcn_wave_barrier();

        // Weighted V on the matrix cores: per V load set and float4 component
        // e, one 4x4x1 MFMA adds p[row][head i] * V[row][4*vj + e] for the
        // four heads of a quad (A: lane 4b+i gives p of head i for its row;
        // B: each lane its own V component).
        // (With PART every probability is read ahead of the products: left in
        // place, each set's read waited for in turn.  Back to back, Llama-3-8B
        // heads ctx 256 5.04 -> 4.88 us, 1000 5.78 -> 5.67; Llama-3.1-405B
        // 13.9 -> 13.5.  Whole-pass launches measured 0-1% slower with it.)
        float pa[GQ][VS];
        if constexpr (MFMA && PART) {
#pragma unroll
            for (int q = 0; q < GQ; q++)
#pragma unroll
                for (int vs = 0; vs < VS; vs++) {
                    const int h = 4 * q + (lane & 3);
                    pa[q][vs] = (h < G) ? p_lds[wave][(vs * RPV + vg) * G + h] : 0.0f;
                }
        }
#pragma unroll
        for (int vs = 0; vs < VS; vs++) {
            const int r = vs * RPV + vg;
            // the load set holding pos (wave-uniform) reads v_new's float4
            // vj across the wave, at this set: its wait for the v_new load,
            // issued last, then holds up only this set's products
            if (pos_here && pos - base >= vs * RPV && pos - base < (vs + 1) * RPV) {
                const float4 vnew = lane_float4(vnew_l, vj);
                if (base + r == pos) {
                    vb[vs] = vnew;
                    if (store_new) *reinterpret_cast<float4 *>(vc + (size_t)(base + r) * kv_dim + 4 * vj) = vnew;
                }
            }
#pragma unroll
            for (int q = 0; q < GQ; q++) {
                if constexpr (MFMA) {
                    const int h = 4 * q + (lane & 3);
                    const float p = PART ? pa[q][vs] : (h < G) ? p_lds[wave][r * G + h] : 0.0f;
                    acc[q][0] = __builtin_amdgcn_mfma_f32_4x4x1f32(p, vb[vs].x, acc[q][0], 0, 0, 0);
                    acc[q][1] = __builtin_amdgcn_mfma_f32_4x4x1f32(p, vb[vs].y, acc[q][1], 0, 0, 0);
                    acc[q][2] = __builtin_amdgcn_mfma_f32_4x4x1f32(p, vb[vs].z, acc[q][2], 0, 0, 0);
                    acc[q][3] = __builtin_amdgcn_mfma_f32_4x4x1f32(p, vb[vs].w, acc[q][3], 0, 0, 0);
                } else {
                    // acc[q][e][i]: head 4q+i at dim 4*vj + e, as the MFMA leaves it
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        if (4 * q + i >= G) continue;
                        const float p = p_lds[wave][r * G + 4 * q + i];
                        acc[q][0][i] += p * vb[vs].x;
                        acc[q][1][i] += p * vb[vs].y;
                        acc[q][2][i] += p * vb[vs].z;
                        acc[q][3][i] += p * vb[vs].w;
                    }
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    tl.mark(kTlLoopEnd);

    // The new token's row after the loop (up to 4 q heads): the wave whose
    // rows hold pos (its v_new load was issued after its rows' loads, and
    // has arrived with them) rotates k_new in lanes L < HD/4 (float4 L, with
    // float4 L of the table row that the prologue staged in this wave's
    // combine buffer), scores it against each head (a dot product per lane,
    // summed over the 16-lane rows with DPP and over the rows with
    // v_readlane: wave-uniform), and adds p = 2^(s - m_ref) and p * v_new to
    // the head's sum (lane 0's share of it, as score_rows_sum reads) and
    // accumulators (lanes vg == 0: V row slot 0 of dims 4*vj .. +3), raising
    // the reference max first if the score exceeds it by kLazyMax.  The
    // heads' chains are independent and laid out step by step, so that they
    // overlap.  The rotated k and v_new go to cache[layer][pos] when the
    // kernel is done with everything else (NewRow), so that the merge's
    // drain does not wait for them.
    if constexpr (NEW_AFTER) {
        if (has_pos && wave == ((pos - chunk_begin) % S::ROWS) / R) {
            float4 krot = make_float4(0.f, 0.f, 0.f, 0.f);
            if (lane < D4) {
                krot = rope4(knew_l, nt_lds[D4 + lane]);
                if (store_new) {
                    nr.k = krot;
                    nr.v = vnew_l;
                    nr.kdst = kc + (size_t)pos * kv_dim + 4 * lane;
                    nr.vdst = vc + (size_t)pos * kv_dim + 4 * lane;
                    nr.on = true;
                }
            }
            float sh[G];
#pragma unroll
            for (int h = 0; h < G; h++) {
                const float4 qv = q_lds[h][lane % D4];
                const float d = qv.x * krot.x + qv.y * krot.y + qv.z * krot.z + qv.w * krot.w;
                sh[h] = (lane < D4) ? d : 0.0f;
            }
#pragma unroll
            for (int h = 0; h < G; h++) sh[h] += dpp<0x128>(sh[h]);  // row_ror:8
#pragma unroll
            for (int h = 0; h < G; h++) sh[h] += dpp<0x124>(sh[h]);  // row_ror:4
#pragma unroll
            for (int h = 0; h < G; h++) sh[h] += dpp<0x122>(sh[h]);  // row_ror:2
#pragma unroll
            for (int h = 0; h < G; h++) sh[h] += dpp<0x121>(sh[h]);  // row_ror:1
            bool grow = false;
#pragma unroll
            for (int h = 0; h < G; h++) {
                // the rows that hold dims: one at head_dim 64, two at 128
                float v = lane_value(sh[h], 0);
#pragma unroll
                for (int row = 1; row < D4 / 16; row++) v += lane_value(sh[h], 16 * row);
                sh[h] = v;
                grow |= sh[h] > m_ref[h] + kLazyMax;
            }
            if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
                for (int h = 0; h < G; h++) {
                    const float m_new = fmaxf(m_ref[h], sh[h]);
                    const float alpha = fast_exp2(m_ref[h] - m_new);
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[h / 4][e][h % 4] *= alpha;
                    l_run[h] *= alpha;
                    m_ref[h] = m_new;
                }
            }
#pragma unroll
            for (int h = 0; h < G; h++) {
                const float p = fast_exp2(sh[h] - m_ref[h]);
                l_run[h] += (lane == 0) ? p : 0.0f;
                const float pv = (vg == 0) ? p : 0.0f;
                acc[h / 4][0][h % 4] += pv * vnew_l.x;
                acc[h / 4][1][h % 4] += pv * vnew_l.y;
                acc[h / 4][2][h % 4] += pv * vnew_l.z;
                acc[h / 4][3][h % 4] += pv * vnew_l.w;
            }
        }
    }

    // Per-wave partials to LDS.
    if constexpr (FLAT) {
        flush();
    } else if constexpr (!PART) {
#pragma unroll
        for (int h = 0; h < G; h++)
            comb_o[wave][vg][h][vj] = make_float4(acc[h / 4][0][h % 4], acc[h / 4][1][h % 4],
                                                  acc[h / 4][2][h % 4], acc[h / 4][3][h % 4]);
    } else
        slot_sums<HD, G>(acc, lane, [&](int, int h, float4 o) { comb_o[wave][0][h][vj] = o; });
#pragma unroll
    for (int h = 0; h < G; h++) {
        const float lw = score_rows_sum(FLAT ? l_sum[h] : l_run[h]);
        if (lane == 0) {
            comb_l[h][wave] = lw;
            comb_m[h][wave] = m_ref[h];
        }
    }
    __syncthreads();
    tl.mark(kTlCombined);

    // Combine the waves: one float4 of one head per thread.
    const bool single = (n_local == 1);
    // (a flat launch's records: those of an XCD's segments together)
    const int n_items = FLAT ? (a.n_groups + kXcds - 1) / kXcds : 0;
    const int n_rec = FLAT ? flat_records(grid_chunks, n_items) : records_per_head(grid_chunks);
    const size_t ws_head0 = (size_t)(FLAT ? xcd : pgroup) * G * (size_t)n_rec;
    const int rec0 = FLAT ? fs.rec0 : 0;                    // the group's first chunk's record
    const int sub_rec0 = FLAT ? flat_sub_record(grid_chunks, n_items, rec0, fs.item) : grid_chunks;  // its first sub-group's
    // A part-group's finished result: the output row (one part), or the
    // part's unnormalised record for the cross-XCD merge launch.
    const bool parts = !FLAT && spread_log2 > 0;
    auto emit = [&](int head, int col, float4 o, float M, float L) {
        if (parts) {
            reinterpret_cast<float4 *>(a.ws_po + ((size_t)pgroup * G + head) * HD)[col] = o;
            if (col == 0) a.ws_pml[(size_t)pgroup * G + head] = make_float2(M, L);
        } else {
            scale4(o, 1.0f / L);
            reinterpret_cast<float4 *>(a.out + (size_t)seq * q_dim + (size_t)(kg.qh0 + head) * HD)[col] = o;
        }
    };
    const uint32_t ws_o_bytes = (uint32_t)(G * n_rec * HD) * 4u;
    const uint32_t ws_ml_bytes = (uint32_t)(G * n_rec) * 8u;
    const __amdgpu_buffer_rsrc_t wo_rsrc = make_rsrc(a.ws_o + ws_head0 * HD, ws_o_bytes);
    const __amdgpu_buffer_rsrc_t wm_rsrc = make_rsrc(a.ws_ml + ws_head0, ws_ml_bytes);
    for (int idx = tid; idx < G * D4; idx += S::THREADS) {
        const int ch = idx / D4, cd4 = idx % D4;  // head, float4 column
        // Every LDS read of this thread as one batch ahead of the arithmetic:
        // left to the compiler, two reads were in flight at a time between
        // the fused multiply-adds, one LDS round trip per wave's partial.
        float mw[NW], lw[NW];
        float4 ow[NW][SLOTS];
#pragma unroll
        for (int w = 0; w < NW; w++) mw[w] = comb_m[ch][w];
#pragma unroll
        for (int w = 0; w < NW; w++)
#pragma unroll
            for (int r = 0; r < SLOTS; r++) ow[w][r] = comb_o[w][r][ch][cd4];
#pragma unroll
        for (int w = 0; w < NW; w++) lw[w] = comb_l[ch][w];
        __builtin_amdgcn_sched_barrier(0);
        float M = -INFINITY, L = 0.f;
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < NW; w++) M = fmaxf(M, mw[w]);
#pragma unroll
        for (int w = 0; w < NW; w++) {
            // (finite: the reference starts at kLowest and only grows)
            const float sc = fast_exp2(mw[w] - M);
#pragma unroll
            for (int r = 0; r < SLOTS; r++) fma4(o, sc, ow[w][r]);
            L += sc * lw[w];
        }
        if (single) {
            emit(ch, cd4, o, M, L);
        } else {
            // Partial o and (max, sum), into this XCD's L2.
            const uint32_t row = (uint32_t)(ch * n_rec + rec0 + lc);
            buf_store4(wo_rsrc, row * (HD * 4u) + 16u * cd4, o);
            if (cd4 == 0) buf_store2(wm_rsrc, row * 8u, make_float2(M, L));
        }
    }
    tl.mark(kTlStored);
    if (single) {
        tl.role(kTlRoleSingle, 0);
        return;
    }

    // Fold records [first, first + n) of the G heads: thread = (head mh < GM,
    // record lane mg, float4 column md4); record lane mg takes records
    // first + mg, first + mg + MG, ... with an online max, eight records of
    // loads in flight at a time, then the record lanes meet in LDS.
    // Leaves (o, M, L) of head mh, columns md4, in the threads with mg == 0.
    // The loads are device-scope (sc1), which always read L2: one 128-byte
    // line holds the (max, sum) records of two sub-groups, and a copy that
    // this CU's L1 took while folding one of them could predate the other's
    // stores.  With G = 3 the threads of the padding head (mh == G) take
    // part in the barriers only: their loads read 0 and they store nothing.
    const int mh = tid / (MG * D4), mg = (tid / D4) % MG, md4 = tid % D4;
    const bool live = mh < G;
    static_assert(sizeof(comb_o) >= sizeof(float4) * GM * MG * D4, "merge scratch");
    static_assert(sizeof(p_lds) >= sizeof(float) * 2 * GM * MG, "merge scratch");
    float4 *mo = &comb_o[0][0][0][0];      // [GM][MG][D4]
    float *mmx = &p_lds[0][0];             // [GM][MG]
    float *mls = &p_lds[0][0] + GM * MG;   // [GM][MG]
    constexpr int B = 8;    // records in flight per lane
    constexpr int BW = 20;  // per lane in the one-level final fold of the asymmetric merge
    // Online fold of records first + c, c = c_begin, c_begin + step, ... < n,
    // into (oo, mm, ll): B records of loads in flight at a time (L2 reads).
    auto fold_lane = [&](int first, int c_begin, int step, int n, float4 &oo, float &mm, float &ll) {
        for (int c0 = c_begin; c0 < n; c0 += step * B) {
            float2 mlb[B];
            float4 ob[B];
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int c = c0 + j * step;
                const uint32_t row = (uint32_t)(mh * n_rec + first + c);
                // past n: an offset at the end of the range reads 0
                const bool in = live && c < n;
                mlb[j] = buf_load2<kSc1>(wm_rsrc, in ? row * 8u : ws_ml_bytes);
                ob[j] = buf_load4<kSc1>(wo_rsrc, in ? row * (HD * 4u) + 16u * md4 : ws_o_bytes);
            }
            float m_new = mm;
#pragma unroll
            for (int j = 0; j < B; j++)
                if (c0 + j * step < n) m_new = fmaxf(m_new, mlb[j].x);
            const float al = (mm == -INFINITY) ? 0.f : fast_exp2(mm - m_new);
            scale4(oo, al);
            ll *= al;
#pragma unroll
            for (int j = 0; j < B; j++) {
                const float w = (c0 + j * step < n) ? fast_exp2(mlb[j].x - m_new) : 0.f;
                fma4(oo, w, ob[j]);
                ll += w * mlb[j].y;
            }
            mm = m_new;
        }
    };
    // Fold records [first, first + n_rt) of the heads [h0, h0 + GH) and emit
    // the heads' results.  GH is a compile-time count: all GM heads, or half
    // of them when two workgroups share the final fold.  The threads are
    // laid out over those heads, with MGH record lanes per head: record lane
    // fg takes records fg, fg + MGH, ... as one batch of loads (n <= MGH * BW
    // a compile-time count, n_rt <= n; records [n_rt, n) read past the range,
    // 0, and count as empty).  With MGH <= 4 a wave holds MGH rows of 16
    // lanes per 16 columns, one row per record lane, so that 16 adjacent
    // lanes read 256 contiguous bytes of one record and the record lanes of
    // a (head, column) meet across rows through the lane crossbar
    // (rows_reduce), without LDS or a barrier; with more record lanes (few
    // heads) they meet in LDS.  (Record
    // lanes in adjacent lanes, with one 16-byte column per record and lane,
    // made the fold's loads four times slower to issue: 0.5-0.8 us at
    // Llama-3-8B.)  The (max, sum) pairs, which the D4 lanes of a record
    // lane all need, are loaded once per (head, record) across the
    // workgroup, ahead of the partial outputs, and shared through LDS (at
    // [head][record], so that the two halves of the heads use disjoint
    // words): a load of each pair in every lane that needs it cost about
    // 0.5 us at Llama-3-8B ctx 4096.
    auto fold_emit = [&](int h0, auto gh_c, int first, auto n_c, int n_rt) {
        constexpr int GH = decltype(gh_c)::value;
        constexpr int n = decltype(n_c)::value;
        constexpr int MGH = S::THREADS / (GH * D4);
        static_assert(MGH * GH * D4 == S::THREADS && D4 % 16 == 0, "fold layout");
        static_assert(n <= MGH * BW && n <= kFinalMax, "records per lane");
        constexpr bool ROWS = MGH <= 4;
        // head - h0, record lane, column
        const int fl = tid / (MGH * D4);
        const int fg = ROWS ? (tid / 16) % MGH : (tid / D4) % MGH;
        const int fd = ROWS ? ((tid / (16 * MGH)) % (D4 / 16)) * 16 + tid % 16 : tid % D4;
        const int fh = h0 + fl;
        const bool flive = fh < G;
        constexpr int BL = (n + MGH - 1) / MGH;
        constexpr int NML = GH * n;
        constexpr int MLT = (NML + S::THREADS - 1) / S::THREADS;
        float2 mlv[MLT];
#pragma unroll
        for (int i = 0; i < MLT; i++) {
            const int t = tid + i * S::THREADS, h = h0 + t / n, c = t % n;
            const bool in = t < NML && h < G && c < n_rt;
            mlv[i] = buf_load2<kSc1>(wm_rsrc, in ? (uint32_t)(h * n_rec + first + c) * 8u : ws_ml_bytes);
        }
        __builtin_amdgcn_sched_barrier(0);
        float4 ob[BL];
#pragma unroll
        for (int j = 0; j < BL; j++) {
            const int c = fg + j * MGH;
            const uint32_t row = (uint32_t)(fh * n_rec + first + c);
            const bool in = flive && c < n_rt;
            ob[j] = buf_load4<kSc1>(wo_rsrc, in ? row * (HD * 4u) + 16u * fd : ws_o_bytes);
        }
        __builtin_amdgcn_sched_barrier(0);
        tl.mark(kTlFoldIssued);
#pragma unroll
        for (int i = 0; i < MLT; i++) {
            const int t = tid + i * S::THREADS;
            if (t < NML) ml_lds[h0 * n + t] = (t % n < n_rt) ? mlv[i] : make_float2(-INFINITY, 0.f);
        }
        __syncthreads();
        tl.mark(kTlFoldLoaded);
        float2 mlb[BL];
#pragma unroll
        for (int j = 0; j < BL; j++) {
            const int c = fg + j * MGH;
            mlb[j] = c < n ? ml_lds[fh * n + c] : make_float2(-INFINITY, 0.f);
        }
        float mm = -INFINITY, ll = 0.f;
        float4 oo = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int j = 0; j < BL; j++)
            if (fg + j * MGH < n) mm = fmaxf(mm, mlb[j].x);
        const float mref = (mm == -INFINITY) ? 0.f : mm;
#pragma unroll
        for (int j = 0; j < BL; j++) {
            const float w = (fg + j * MGH < n) ? fast_exp2(mlb[j].x - mref) : 0.f;
            fma4(oo, w, ob[j]);
            ll += w * mlb[j].y;
        }
        if constexpr (ROWS) {
            // The record lanes meet across rows: max, rescale, sums.
            const float Mx = rows_reduce<MGH, true>(mm);
            const float sc = (mm == -INFINITY) ? 0.f : fast_exp2(mm - Mx);
            const float4 ox =
                make_float4(rows_reduce<MGH, false>(sc * oo.x), rows_reduce<MGH, false>(sc * oo.y),
                            rows_reduce<MGH, false>(sc * oo.z), rows_reduce<MGH, false>(sc * oo.w));
            const float Lx = rows_reduce<MGH, false>(sc * ll);
            if (fg == 0 && flive) emit(fh, fd, ox, Mx, Lx);
            tl.mark(kTlFolded);
        } else {
            __syncthreads();  // LDS scratch is free
            mo[(fl * MGH + fg) * D4 + fd] = oo;
            if (fd == 0) {
                mmx[fl * MGH + fg] = mm;
                mls[fl * MGH + fg] = ll;
            }
            __syncthreads();
            if (fg == 0 && flive) {
                float Mx = -INFINITY;
#pragma unroll
                for (int g = 0; g < MGH; g++) Mx = fmaxf(Mx, mmx[fl * MGH + g]);
                float Lx = 0.f;
                float4 ox = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int g = 0; g < MGH; g++) {
                    const float mgv = mmx[fl * MGH + g];
                    const float sc = (mgv == -INFINITY) ? 0.f : fast_exp2(mgv - Mx);
                    fma4(ox, sc, mo[(fl * MGH + g) * D4 + fd]);
                    Lx += sc * mls[fl * MGH + g];
                }
                emit(fh, fd, ox, Mx, Lx);
            }
            tl.mark(kTlFolded);
        }
    };
    // Fold records [first, first + n) of the G heads into (ox, Mx, Lx) of
    // the threads with mg == 0.  Up to B records are one batch of loads in
    // those threads alone; more are spread over the MG record lanes, which
    // then meet in LDS.
    auto fold = [&](int first, int n, float4 &ox, float &Mx, float &Lx) {
        if (n <= B) {
            if (mg == 0) {
                ox = make_float4(0.f, 0.f, 0.f, 0.f);
                Mx = -INFINITY;
                Lx = 0.f;
                fold_lane(first, 0, 1, n, ox, Mx, Lx);
            }
            return;
        }
        float mm = -INFINITY, ll = 0.f;
        float4 oo = make_float4(0.f, 0.f, 0.f, 0.f);
        fold_lane(first, mg, MG, n, oo, mm, ll);
        __syncthreads();  // LDS scratch is free (combine buffers / earlier fold)
        mo[(mh * MG + mg) * D4 + md4] = oo;
        if (md4 == 0) {
            mmx[mh * MG + mg] = mm;
            mls[mh * MG + mg] = ll;
        }
        __syncthreads();
        if (mg == 0) {
            Mx = -INFINITY;
#pragma unroll
            for (int g = 0; g < MG; g++) Mx = fmaxf(Mx, mmx[mh * MG + g]);
            Lx = 0.f;
            ox = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int g = 0; g < MG; g++) {
                const float mgv = mmx[mh * MG + g];
                const float sc = (mgv == -INFINITY) ? 0.f : fast_exp2(mgv - Mx);
                fma4(ox, sc, mo[(mh * MG + g) * D4 + md4]);
                Lx += sc * mls[mh * MG + g];
            }
        }
    };
    int *ctr = a.counters + (size_t)pgroup * (size_t)counters_per_group(grid_chunks);

    // The fold of a one-level merge's records [first, first + n_rt) (n_c a
    // compile-time bound), after this workgroup counted in with result prev.
    // The last arrival folds.  From kHelpMinRecords records on (G > 1) the
    // heads are folded in two halves, and with the helper on (a.merge_asym
    // >> 1) the second-to-last arrival waits for the last (fold_helper_wait)
    // and folds the second half: that halves the bytes the last arrival's CU
    // takes in, and a fold's time grows by about 24 ns per 2 KiB record at
    // Llama-3-8B.
    auto final_fold = [&](int first, auto n_c, int n_rt, int prev) {
        if constexpr (GM >= 2) {
            if (n_rt >= kHelpMinRecords) {
                // The two halves of the heads are folded with the same
                // layout whoever folds them, so the result does not depend
                // on the helper.
                constexpr auto gh = std::integral_constant<int, GM / 2>{};
                const int help = a.merge_asym >> 1;
                if (help && prev == n_rt - 2) {
                    __syncthreads();  // every thread has read s_last
                    if (tid == 0) s_last = fold_helper_wait(ctr, n_rt, help);
                    __syncthreads();
                    tl.role(kTlRoleHelper, prev);
                    if (s_last) fold_emit(GM / 2, gh, first, n_c, n_rt);
                    return;
                }
                if ((prev & (kGiveUp - 1)) != n_rt - 1) return;
                tl.role(kTlRoleFinal, prev);
                fold_emit(0, gh, first, n_c, n_rt);
                if (help && prev < kGiveUp) return;  // the helper folds the other half
                if (tid == 0) ctr[0] = 0;
                fold_emit(GM / 2, gh, first, n_c, n_rt);
                return;
            }
        }
        if ((prev & (kGiveUp - 1)) != n_rt - 1) return;
        tl.role(kTlRoleFinal, prev);
        if (tid == 0) ctr[0] = 0;
        fold_emit(0, std::integral_constant<int, GM>{}, first, n_c, n_rt);
    };
    // The asymmetric merge (see the header), for NC chunks: chunks [0, NC/2)
    // fold in sub-groups whose records go right after the chunk records, and
    // the final fold reads records [NC/2, NC + NC/2/kSubGroup), one range.
    // NC is compiled in (32, 48 or 64) so that the final fold's loads are
    // exact.
    auto merge_asym = [&](auto nc_c) {
        constexpr int NC = decltype(nc_c)::value, half = NC / 2, n_final = half + half / kSubGroup;
        if (lc < half) {
            const int sg1 = lc / kSubGroup;
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            tl.mark(kTlDrained);
            if (tid == 0) {
                const int prev = __hip_atomic_fetch_add(ctr + (1 + sg1) * kCtrStride, 1, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP);
                s_last = (prev == kSubGroup - 1);
            }
            __syncthreads();
            tl.mark(kTlSubCounted);
            if (!s_last) return;
            tl.role(kTlRoleSub, 0);
            if (tid == 0) ctr[(1 + sg1) * kCtrStride] = 0;
            float4 o1;
            float M1, L1;
            fold(sg1 * kSubGroup, kSubGroup, o1, M1, L1);
            if (mg == 0 && live) {
                const uint32_t row = (uint32_t)(mh * n_rec + NC + sg1);
                buf_store4(wo_rsrc, row * (HD * 4u) + 16u * md4, o1);
                if (md4 == 0) buf_store2(wm_rsrc, row * 8u, make_float2(M1, L1));
            }
            tl.mark(kTlSubFolded);
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (lc >= half) tl.mark(kTlDrained);
        if (tid == 0) s_last = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
        tl.mark(kTlCounted);
        const int prev = s_last;
        final_fold(half, std::integral_constant<int, n_final>{}, n_final, prev);
    };
    // One level for launches without the asymmetric shape and 2-40 chunks:
    // every chunk counts into the final counter and the last folds all
    // records as one batch of loads, compiled for NC = n_local rounded up to
    // a multiple of 8 (the records past n_local are empty).  Against the
    // two-level tree (sub-groups of 8, then their records) this leaves out a
    // store, drain and atomic round trip for 8-40 KiB more loads into the
    // last CU: Llama-3-8B ctx 1024 8.03 -> 6.77 us, ctx 2048 8.33 -> 7.58 us.
    // Up to 8 chunks it replaces a fold in the threads of one record lane,
    // which loaded each (max, sum) pair in every lane: ctx 256 6.60 -> 6.52.
    auto merge_flat = [&](auto nc_c) {
        constexpr int NC = decltype(nc_c)::value;
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        tl.mark(kTlDrained);
        if (tid == 0) s_last = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
        tl.mark(kTlCounted);
        const int prev = s_last;
        final_fold(rec0, std::integral_constant<int, NC>{}, n_local, prev);
    };
    if (!(a.merge_asym & 1) && n_local > 1) {
        if (n_local <= 8) return merge_flat(std::integral_constant<int, 8>{});
        if constexpr (16 <= MG * BW) {
            if (n_local <= 16) return merge_flat(std::integral_constant<int, 16>{});
        }
        if constexpr (24 <= MG * BW) {
            if (n_local <= 24) return merge_flat(std::integral_constant<int, 24>{});
        }
        if constexpr (32 <= MG * BW) {
            if (n_local <= 32) return merge_flat(std::integral_constant<int, 32>{});
        }
        if constexpr (40 <= MG * BW) {
            if (n_local <= 40) return merge_flat(std::integral_constant<int, 40>{});
        }
    }
    if (!FLAT && (a.merge_asym & 1)) {
        if constexpr (32 + 4 <= MG * BW) {
            if (n_local == 64) return merge_asym(std::integral_constant<int, 64>{});
        }
        if constexpr (24 + 3 <= MG * BW) {
            if (n_local == 48) return merge_asym(std::integral_constant<int, 48>{});
        }
        if constexpr (16 + 2 <= MG * BW) {
            if (n_local == 32) return merge_asym(std::integral_constant<int, 32>{});
        }
    }

    // Level 1: once this workgroup's partials have reached L2 (stores
    // drained), count it in on its sub-group's counter (an L2 atomic).
    const int sg = lc / kSubGroup;
    const int n_sg = (n_local + kSubGroup - 1) / kSubGroup;
    const int sg_n = min(kSubGroup, n_local - sg * kSubGroup);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    tl.mark(kTlDrained);
    if (tid == 0) {
        const int prev = __hip_atomic_fetch_add(ctr + (1 + sg) * kCtrStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        s_last = (prev == sg_n - 1);
    }
    __syncthreads();
    tl.mark(kTlSubCounted);
    if (!s_last) return;
    tl.role(kTlRoleSub, 0);
    if (tid == 0) ctr[(1 + sg) * kCtrStride] = 0;
    float4 ox;
    float Mx, Lx;
    fold(rec0 + sg * kSubGroup, sg_n, ox, Mx, Lx);
    if (n_sg == 1) {
        if (mg == 0 && live) emit(mh, md4, ox, Mx, Lx);
        tl.role(kTlRoleFinal, 0);
        tl.mark(kTlFolded);
        return;
    }
    if (mg == 0 && live) {
        const uint32_t row = (uint32_t)(mh * n_rec + sub_rec0 + sg);
        buf_store4(wo_rsrc, row * (HD * 4u) + 16u * md4, ox);
        if (md4 == 0) buf_store2(wm_rsrc, row * 8u, make_float2(Mx, Lx));
    }

    // Level 2: the last sub-group to finish folds the sub-group records.
    tl.mark(kTlSubFolded);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
        const int prev = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        s_last = (prev == n_sg - 1);
    }
    __syncthreads();
    tl.mark(kTlCounted);
    if (!s_last) return;
    tl.role(kTlRoleFinal, n_sg - 1);
    if (tid == 0) ctr[0] = 0;
    fold(sub_rec0, n_sg, ox, Mx, Lx);
    if (mg == 0 && live) emit(mh, md4, ox, Mx, Lx);
    tl.mark(kTlFolded);
}

template <int HD, int G, int NW, bool MFMA = true, bool PART = false, int KVS = 0>
__global__ __launch_bounds__(NW * kWave, (MFMA && G == 8 && HD == 128) ? 2 : 1) void decode_attention_kernel(LEAP_PRELOAD_PARAMS, StepArgs a)
{
    Timeline tl;
    tl.mark(kTlStart);
    NewRow nr;
    nr.on = false;
    decode_attention_body<HD, G, NW, MFMA, PART, KVS>(a, LEAP_PRELOAD, tl, nr);
    if (nr.on) {
        *reinterpret_cast<float4 *>(nr.kdst) = nr.k;
        *reinterpret_cast<float4 *>(nr.vdst) = nr.v;
    }
#ifdef LEAP_TIMELINE
    tl.mark(kTlEnd);
    tl.flush(a.tl);
#endif
}

// Inclusive prefix sum over the 64 lanes of a wave (DPP: within the 16-lane
// rows, then row 0 into row 1 and row 2 into row 3, then the lower half into
// the upper).
__device__ __forceinline__ int wave_prefix_sum(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31
    return v;
}

// The decode kernel for a batch whose groups do not cut evenly over the CUs
// (see kFlatSegmentRows; the host's rule: flat_launch).  StepArgs::grid_chunks
// is the workgroups per XCD, StepArgs::chunk the rows that an item's start
// counts as; at most kFlatMaxItems items per XCD.
// What bounds it is the CU with the most to take in, then the merge.  Graph
// replay, us per launch, uniform chunks (at the host's choice) -> flat:
// Llama-3-8B heads, 16 sequences of 200-2000 rows 33.3 -> 29.2 (145 MB, 4.35
// -> 4.96 TB/s), 8 of them 23.2 -> 18.0, 6 of 400-4000 rows 29.2 -> 24.1, 64
// of 400-4000 189.5 -> 175.2; 12 sequences of 2000 rows 46.9 -> 37.3 and of
// 8000 164.7 -> 122.5; Llama-3-70B heads, 16 of 200-2000 rows 45.3 -> 32.2;
// TinyLlama heads, 64 of 200-2000 rows 50.7 -> 33.2.
template <int HD, int G, int NW, int KVS>
__global__ __launch_bounds__(NW * kWave, (G == 8 && HD == 128) ? 2 : 1) void decode_attention_flat_kernel(LEAP_PRELOAD_PARAMS, StepArgs a)
{
    Timeline tl;
    tl.mark(kTlStart);
    const int xcd = blockIdx.x % kXcds, w = blockIdx.x / kXcds;
    __shared__ int2 items_lds[NW][kWave];  // per wave: each item's rows and the rows up to its end
    asm volatile("" ::"s"(a.pos_dev), "s"(a.max_pos), "s"(a.seq_len), "s"(a.n_groups), "s"(a.grid_chunks),
                 "s"(a.chunk), "s"(a.by_kv_heads.m), "s"(a.by_kv_heads.s), "s"(a.by_grid_chunks.m),
                 "s"(a.by_grid_chunks.s));
    const int n_wg = a.grid_chunks, start_rows = a.chunk;
    const int n_items = (a.n_groups - xcd + kXcds - 1) / kXcds;
    int at, stop, run;
    {
        // Every wave works out the XCD's rows and the workgroup's run by
        // itself: lane i has item i's rows, 0 for a position the launch
        // cannot serve.
        const int i = threadIdx.x % kWave;
        int rows = 0;
        if (i < n_items) {
            const int pos = a.pos_dev[fast_div((uint32_t)(i * kXcds + xcd), a.by_kv_heads)];
            if (pos >= 0 && pos < a.seq_len && pos <= a.max_pos) rows = pos + 1 + start_rows;
        }
        const int upto = wave_prefix_sum(rows);
        const int total = __builtin_amdgcn_readlane(upto, kWave - 1);
        run = max((int)fast_div((uint32_t)(total + n_wg - 1), a.by_grid_chunks), kFlatMinRun);
        at = w * run;
        stop = min(at + run, total);
        items_lds[threadIdx.x / kWave][i] = make_int2(rows, upto);
        // The output rows of a sequence whose position the launch cannot
        // serve read NaN (item i by workgroup i mod n_wg).
        for (uint64_t bad = __builtin_amdgcn_ballot_w64(i < n_items && rows == 0); bad; bad &= bad - 1) {
            const int item = __builtin_ctzll(bad);
            if (item % n_wg != w) continue;
            const int group = item * kXcds + xcd, seq = (int)fast_div((uint32_t)group, a.by_kv_heads);
            const int kvv = group - seq * a.n_kv_heads;
            const int qh0 = KVS ? kv_group<G>(kvv, a.n_kv_heads, KVS).qh0 : kvv * G;
            for (int j = threadIdx.x; j < G * HD; j += NW * kWave)
                a.out[(size_t)seq * a.n_heads * HD + (size_t)qh0 * HD + j] = __builtin_nanf("");
        }
    }
    while (at < stop) {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int2 it = items_lds[tid / kWave][tid % kWave];
        // the item that row `at` counts in: the first to end past it
        const int item = __builtin_ctzll(__builtin_amdgcn_ballot_w64(it.y > at));
        const int item_end = __builtin_amdgcn_readlane(it.y, item);
        const FlatSegment fs = flat_segment(w, run, at, stop, item, item_end - __builtin_amdgcn_readlane(it.x, item),
                                            item_end, start_rows);
        at = item_end;
        if (fs.begin == fs.end) continue;
        NewRow nr;
        nr.on = false;
        // (the arguments are read again for each segment, rather than held in
        // scalar registers through the ones before)
        const StepArgs la = late_args(a, kArgsOffset);
        const Preload pre{la.q, la.k_new, la.k_cache, la.v_cache, la.rope, 0u,
                          (uint32_t)la.grid_chunks | ((uint32_t)la.n_kv_heads << 16), 0u, 0u};
        decode_attention_body<HD, G, NW, true, true, KVS, true>(la, pre, tl, nr, fs);
        if (nr.on) {
            *reinterpret_cast<float4 *>(nr.kdst) = nr.k;
            *reinterpret_cast<float4 *>(nr.vdst) = nr.v;
        }
        __syncthreads();  // the workgroup's LDS is free
    }
#ifdef LEAP_TIMELINE
    tl.mark(kTlEnd);
    tl.flush(a.tl);
#endif
}

// The cross-XCD merge of a spread launch: after the decode launch, the parts
// of each (sequence, KV head) group have left one unnormalised record each
// (the launch boundary makes them visible to every XCD).  One workgroup per
// group, one thread per (q head, float4 column): fold the group's non-empty
// parts in part order with an online max, normalise, write the output row.
template <int HD, int G>
__global__ __launch_bounds__(G * HD / 4) void part_merge_kernel(StepArgs a)
{
    constexpr int D4 = HD / 4;
    // the argument block as one batch of loads, as in the decode kernel
    asm volatile("" ::"s"(a.pos_dev), "s"(a.ws_po), "s"(a.ws_pml), "s"(a.out), "s"(a.pos_scalar), "s"(a.max_pos),
                 "s"(a.seq_len), "s"(a.n_heads), "s"(a.n_kv_heads), "s"(a.chunk), "s"(a.grid_chunks),
                 "s"(a.n_groups), "s"(a.spread_log2), "s"(a.even_chunks), "s"(a.kv_split));
    const int group = blockIdx.x;
    if (group >= a.n_groups) return;
    const int seq = group / a.n_kv_heads;
    const KvGroup kg = kv_group<G>(group % a.n_kv_heads, a.n_kv_heads, a.kv_split);
    const int pos = a.pos_dev ? a.pos_dev[seq] : a.pos_scalar;
    const int q_dim = a.n_heads * HD;
    if (pos < 0 || pos >= a.seq_len || pos > a.max_pos) {
        // a position the launch cannot serve: the output rows read NaN
        for (int i = threadIdx.x; i < G * HD; i += G * HD / 4)
            a.out[(size_t)seq * q_dim + (size_t)kg.qh0 * HD + i] = __builtin_nanf("");
        return;
    }
    const int n_chunks = seq_chunks(a, pos + 1);
    const int n_parts = min(1 << a.spread_log2, (n_chunks + a.grid_chunks - 1) / a.grid_chunks);
    const int h = threadIdx.x / D4, c = threadIdx.x % D4;
    const size_t pg0 = (size_t)group << a.spread_log2;
    float M = -INFINITY;
    for (int p = 0; p < n_parts; p++) M = fmaxf(M, a.ws_pml[(pg0 + p) * G + h].x);
    float L = 0.f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p = 0; p < n_parts; p++) {
        const float2 ml = a.ws_pml[(pg0 + p) * G + h];
        const float w = (ml.x == -INFINITY) ? 0.f : fast_exp2(ml.x - M);
        fma4(o, w, reinterpret_cast<const float4 *>(a.ws_po + ((pg0 + p) * G + h) * HD)[c]);
        L += w * ml.y;
    }
    scale4(o, 1.0f / L);
    reinterpret_cast<float4 *>(a.out + (size_t)seq * q_dim + (size_t)(kg.qh0 + h) * HD)[c] = o;
}

// ---- launch and stream floors (measurement only) ----------------------------
//
// Two kernels with the decode kernel's grid, block size and arguments (the
// preloaded words and the argument block), for measuring what any
// one-launch design at a given shape must pay:
//   - floor_launch_kernel reads two kernel arguments and exits (the launch,
//     the preload and the drain of an empty grid);
//   - floor_stream_kernel streams the same K and V rows with the same loads
//     (128-bit, non-temporal, the same lane layout and passes) and only sums
//     them (the launch plus the bare stream of the step's bytes).
// Neither writes anything: the sums are kept only behind a test that real
// data never meets (a NaN with a particular payload).

template <int HD, int G, int NW>
__global__ __launch_bounds__(NW * kWave) void floor_launch_kernel(LEAP_PRELOAD_PARAMS, StepArgs a)
{
    if (pre_w0 == 0u && pre_w1 == 0u) a.out[threadIdx.x] = 0.0f;
}

template <int HD, int G, int NW, int KVS, bool PART>
__global__ __launch_bounds__(NW * kWave) void floor_stream_kernel(LEAP_PRELOAD_PARAMS, StepArgs a)
{
    using S = Shape<HD, G, NW>;
    constexpr int NF = S::NF, R = S::R, KS = S::KS, LPV = S::LPV, RPV = S::RPV, VS = S::VS;
    // The prologue as the decode kernel's: from the preloaded words for one
    // sequence at a host position, else from the argument block.  (The
    // floors run without a spread.)
    const int xcd = blockIdx.x % kXcds;
    const int local = blockIdx.x / kXcds;
    const int grid_chunks = (int)(pre_w0 & 1023u);
    const int n_kv_heads = (int)(pre_w0 >> 16);
    const int lq = (int)fast_div((uint32_t)local, FastDiv{pre_m_gc, (pre_w0 >> 10) & 15u});
    const int chunk_id = local - lq * grid_chunks;
    const int group = lq * kXcds + xcd;
    int seq, pos, n_chunks, cq, cr;
    size_t slab;
    if (pre_w1 != kPreGeneral) {
        if (group >= n_kv_heads) return;
        seq = 0;
        pos = (int)(pre_w1 & (kPreLimit - 1));
        n_chunks = (int)(pre_w1 >> 21);
        cq = (int)(pre_w2 & (kPreLimit - 1));
        cr = (int)(pre_w2 >> 21);
        slab = 0;
    } else {
        asm volatile("" ::"s"(a.pos_dev), "s"(a.seq_stride), "s"(a.pos_scalar), "s"(a.max_pos), "s"(a.seq_len),
                     "s"(a.chunk), "s"(a.n_groups), "s"(a.even_chunks), "s"(a.by_kv_heads.m), "s"(a.by_kv_heads.s),
                     "s"(a.by_chunk.m), "s"(a.by_chunk.s), "s"(a.by_even.m), "s"(a.by_even.s));
        if (group >= a.n_groups) return;
        seq = (int)fast_div((uint32_t)group, a.by_kv_heads);
        pos = a.pos_dev ? a.pos_dev[seq] : a.pos_scalar;
        if (pos < 0 || pos >= a.seq_len || pos > a.max_pos) return;
        n_chunks = seq_chunks(a, pos + 1);
        if (a.even_chunks > 0) {
            cq = pos + 1 >= a.even_chunks ? (int)fast_div((uint32_t)(pos + 1), a.by_even) : 1;
            cr = pos + 1 - cq * n_chunks;
        } else {
            cq = a.chunk;
            cr = 0;
        }
        slab = (size_t)seq * (size_t)a.seq_stride;
    }
    const int kvh = kv_group<G>(group - seq * n_kv_heads, n_kv_heads, KVS).kvh;
    const int T = pos + 1;
    if (chunk_id >= n_chunks) return;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const uint32_t row_bytes = (uint32_t)((n_kv_heads >> KVS) * HD) * 4u;
    const int chunk_begin = min(chunk_id * cq + min(chunk_id, cr), T);
    const int chunk_end = min((chunk_id + 1) * cq + min(chunk_id + 1, cr), T);
    const uint32_t range = (uint32_t)min(pos, chunk_end) * row_bytes;  // as the step's
    const __amdgpu_buffer_rsrc_t k_rsrc = make_rsrc(pre_k_cache + slab + (size_t)kvh * HD, range);
    const __amdgpu_buffer_rsrc_t v_rsrc = make_rsrc(pre_v_cache + slab + (size_t)kvh * HD, range);
    const int kj = lane & 3, ksl = (lane >> 2) & 7, kq = lane >> 5, krow = 4 * kq + kj;
    const int vg = lane / LPV, vj = lane % LPV;
    const int n_sub = (chunk_end - chunk_begin + S::ROWS - 1) / S::ROWS;
    float sum = 0.0f;
    // passes and skips as the step (PART: the step's instance kind)
    constexpr bool part = PART;
    const int sub0 = (part && n_sub > 1) ? chunk_id % n_sub : 0;
    for (int i = 0; i < n_sub; i++) {
        const int sub = sub0 + i < n_sub ? sub0 + i : sub0 + i - n_sub;
        const int base = chunk_begin + (sub * NW + wave) * R;
        if (part && i > 0 && base >= chunk_end) continue;
        float4 kb[KS][NF], vb[VS];
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int f = 0; f < NF; f++)
                kb[ks][f] = buf_load4<kNt>(k_rsrc, (uint32_t)(base + ks * 8 + krow) * row_bytes + 16u * (uint32_t)(8 * f + ksl));
#pragma unroll
        for (int vs = 0; vs < VS; vs++)
            vb[vs] = buf_load4<kNt>(v_rsrc, (uint32_t)(base + vs * RPV + vg) * row_bytes + 16u * (uint32_t)vj);
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int f = 0; f < NF; f++) sum += kb[ks][f].x + kb[ks][f].y + kb[ks][f].z + kb[ks][f].w;
#pragma unroll
        for (int vs = 0; vs < VS; vs++) sum += vb[vs].x + vb[vs].y + vb[vs].z + vb[vs].w;
    }
    if (__builtin_bit_cast(unsigned, sum) == 0x7FC0DEADu) a.out[threadIdx.x] = sum;
}

}  // namespace leap
