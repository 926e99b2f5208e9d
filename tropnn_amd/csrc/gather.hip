// Staged PairwiseLinear forward for gfx950: the large-batch path of callers
// that lend the forward a workspace. A route kernel writes every item's LUT
// row codes, packed four to a word, and one of two gather kernels sums the
// LUT rows they name out of LDS. Both gathers read each LUT row from memory
// once per workgroup instead of once per (item, table), so a large batch is
// bound by LDS reads rather than by the L2 row gather of the kernels that
// route and gather in one launch (forward.hip), which serve small batches and
// callers without a workspace.
//
// Reference semantics: layers/pairwise.py:127-135 (route), 99-125 (gather),
// layers/base.py:76-77 (scale), as in forward.hip; codes, margins and route
// records are bit-identical to that file's kernels.
#include <algorithm>
#include <type_traits>

#include "device.hpp"
#include "launch.hpp"

namespace tropnn {
namespace {

// Tables are summed in blocks of `per` <= kBlockTables consecutive tables,
// then the blocks in order: the association of the forward.hip kernels, so
// the slice gather's outputs equal theirs bit for bit. The codes of a block
// take kBlockWords words per item whatever `per` is (byte u of the block's 16
// is table block * per + u; bytes past the block's tables are zero).
constexpr int kBlockTables = 16;
constexpr int kBlockWords = kBlockTables / 4;
constexpr int kGatherMinItems = 256;
constexpr long long kStreamMinLut = 32ll << 20;
constexpr int kGatherCus = 256;              // gfx950 (MI355X)
constexpr int kSliceLds = 156 * 1024;        // a CU's LDS for staged slices
constexpr int kRouteLds = 78 * 1024;         // a route workgroup's LDS: two workgroups per CU
constexpr int kSliceIpt = 4;                 // items per thread held across stages

// ------------------------------------------------------------------ route

struct RouteWordsArgs {
    const float *x;
    const int64_t *anchors;
    const float *thr;
    uint32_t *words;  // [groups][pitch]: word g of item b = its codes at positions 4 g .. 4 g + 3
    uint64_t *rec;
    int64_t *indices;
    float *margins;
    uint8_t *codes;
    int items, in_f, tables, comps;
    int per, groups, pitch;
    int bias_mask;           // stream gather: the table's group in its stage ((t >> 2) & mask) rides above the code's bits
    int quads;               // groups of four items per workgroup
    int table_threads, parts;  // thread = part * table_threads + table
    int code_off, rec_off;   // LDS byte offsets (rec_off 0: records stored directly)
    int rec_vec;             // runs of four records start on 16-byte boundaries
};

constexpr int kRouteWordsThreads = 512;  // at most

// One workgroup routes 4 * quads consecutive items. Their input rows lie in
// LDS with four items interleaved, so one 16-byte read gives a feature of four
// items. Thread (part, table) takes its table's comparators once, before the
// rows are staged, and the quads part, part + parts, ...; codes and records
// are gathered in LDS and leave as runs of consecutive items.
template <bool TRAIN, bool DEBUG>
__global__ __launch_bounds__(kRouteWordsThreads) void pairwise_route_words_kernel(RouteWordsArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    using f32x4 = vec_t<float, 4>;
    f32x4 *xs = reinterpret_cast<f32x4 *>(lds);  // [quads][in_f] x 4 items
    uint8_t *cs = lds + a.code_off;              // [4 quads][groups * 4]
    uint64_t *rs = reinterpret_cast<uint64_t *>(lds + a.rec_off);  // [tables][4 quads + 1]
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int NI = 4 * a.quads, C = a.comps, T = a.tables;
    const int b0 = xcd_block_unit(blockIdx.x, gridDim.x) * NI;  // runs of adjacent blocks share lines
    const int n = min(NI, a.items - b0);
    const int part = tid / a.table_threads, t_first = tid - part * a.table_threads;
    int ia[TROPNN_MAX_COMPARISONS], ib[TROPNN_MAX_COMPARISONS];
    float th[TROPNN_MAX_COMPARISONS];
    auto comparators = [&](int t) {
#pragma unroll
        for (int c = 0; c < TROPNN_MAX_COMPARISONS; ++c) {  // loads issued unconditionally
            const size_t k = static_cast<size_t>(min(t, T - 1)) * C + (c < C ? c : 0);
            ia[c] = clamp_index(a.anchors[2 * k], a.in_f);
            ib[c] = clamp_index(a.anchors[2 * k + 1], a.in_f);
            th[c] = a.thr[k];
        }
    };
    const int code_words = NI * a.groups;
    // (positions past the last table keep the bias alone: a row of zeros)
    for (int k = tid; k < code_words; k += nthr)
        reinterpret_cast<uint32_t *>(cs)[k] = static_cast<uint32_t>((k % a.groups) & a.bias_mask) * (0x01010101u << C);
    comparators(t_first);
    for (int q = 0; q < a.quads; ++q) {
        // rows past the last item repeat it: loaded, never stored
        const float *r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = a.x + static_cast<size_t>(min(b0 + 4 * q + i, a.items - 1)) * a.in_f;
#pragma unroll 2
        for (int f = tid; f < a.in_f; f += nthr) xs[q * a.in_f + f] = f32x4{r[0][f], r[1][f], r[2][f], r[3][f]};
    }
    __syncthreads();
    const float inv_per = 1.0f / static_cast<float>(a.per);
    auto position = [&](int t) { return a.per == kBlockTables ? t : t + (kBlockTables - a.per) * small_div(t, inv_per); };
    for (int t = t_first; t < T; t += a.table_threads) {
        if (t != t_first) comparators(t);
        const int pos = position(t);
        const uint32_t bias = static_cast<uint32_t>((t >> 2) & a.bias_mask) << C;
        for (int q = part; q < a.quads; q += a.parts) {
            uint32_t code[4] = {0u, 0u, 0u, 0u}, key[4], pick[4] = {0u, 0u, 0u, 0u};
            float pm[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) key[i] = 0xFFFFFFFFu;
            const f32x4 *xq = xs + q * a.in_f;
#pragma unroll
            for (int c = 0; c < TROPNN_MAX_COMPARISONS; ++c) {
                if (c < C) {  // uniform
                    const f32x4 xa = xq[ia[c]], xb = xq[ib[c]];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float m = (xa[i] - xb[i]) - th[c];
                        code[i] |= (m > 0.f ? 1u : 0u) << c;
                        if constexpr (TRAIN) {
                            // argmin |m|: NaN first, then the smaller magnitude, then the lower index
                            const float mag = fabsf(m);
                            const uint32_t k = mag != mag ? 0u : __builtin_bit_cast(uint32_t, mag) + 1u;
                            if (k < key[i]) {
                                key[i] = k;
                                pick[i] = c;
                                pm[i] = m;
                            }
                        }
                        if constexpr (DEBUG) {
                            if (a.margins != nullptr && 4 * q + i < n)
                                a.margins[(static_cast<size_t>(b0 + 4 * q + i) * T + t) * C + c] = m;
                        }
                    }
                }
            }
            uint64_t rec[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int it = 4 * q + i;
                cs[it * (a.groups * 4) + pos] = static_cast<uint8_t>(code[i] + bias);
                rec[i] = static_cast<uint64_t>(__builtin_bit_cast(uint32_t, pm[i])) | (static_cast<uint64_t>(code[i]) << 32) |
                         (static_cast<uint64_t>(pick[i]) << 48);
            }
            if constexpr (TRAIN) {
                uint64_t *dst = a.rec + static_cast<size_t>(t) * a.items + b0 + 4 * q;
                if (a.rec_off != 0) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) rs[t * (NI + 1) + 4 * q + i] = rec[i];  // + 1: a wave's stores spread over the banks
                } else if (a.rec_vec && 4 * q + 4 <= n) {
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        reinterpret_cast<vec_t<uint64_t, 2> *>(dst)[h] = vec_t<uint64_t, 2>{rec[2 * h], rec[2 * h + 1]};
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (4 * q + i < n) dst[i] = rec[i];
                }
            }
        }
    }
    __syncthreads();
    const int ni_log2 = 31 - __builtin_clz(NI);  // NI is 4, 8 or 16
    for (int k = tid; k < code_words; k += nthr) {
        const int g = k >> ni_log2, i = k & (NI - 1);
        if (i < n)
            a.words[static_cast<size_t>(g) * a.pitch + b0 + i] = reinterpret_cast<const uint32_t *>(cs)[i * a.groups + g];
    }
    if (b0 + n == a.items)  // the pitch's padding names row 0
        for (int k = tid; k < a.groups * (a.pitch - a.items); k += nthr) {
            const int g = k / (a.pitch - a.items), i = k - g * (a.pitch - a.items);
            a.words[static_cast<size_t>(g) * a.pitch + a.items + i] = 0u;
        }
    if constexpr (TRAIN) {
        if (a.rec_off != 0)
            for (int k = tid; k < T * NI; k += nthr) {
                const int t = k >> ni_log2, i = k & (NI - 1);
                if (i < n) a.rec[static_cast<size_t>(t) * a.items + b0 + i] = rs[t * (NI + 1) + i];
            }
    }
    if constexpr (DEBUG) {
        const uint32_t code_mask = (1u << C) - 1u;
        for (int i = 0; i < n; ++i) {
            const size_t row = static_cast<size_t>(b0 + i) * T;
            for (int t = tid; t < T; t += nthr) {
                const uint8_t code = static_cast<uint8_t>(cs[i * (a.groups * 4) + position(t)] & code_mask);
                if (a.indices != nullptr) a.indices[row + t] = code;
                if (a.codes != nullptr) a.codes[row + t] = code;
            }
        }
    }
}

// ------------------------------------------------------------------ slice gather

struct SliceArgs {
    const void *lut;
    const uint32_t *words;
    float *out;
    float scale;
    uint32_t lut_bytes;
    int items, out_f, tables, rows, row_bytes;
    int per, blocks, pitch;      // blocks of `per` tables
    int nblk, block_items;       // workgroups: column slices x item blocks
    int stage_blocks, stages;    // blocks of tables in LDS at a time
    int zero_off;                // LDS byte offset of 16 zero bytes
    int out_vec;                 // rows of out are 16-byte aligned
};

constexpr int kSliceBytes = 16;

// acc += the elements of a 16-byte row piece.
template <typename T>
__device__ __forceinline__ void add_piece(float (&acc)[kSliceBytes / sizeof(T)], const vec_t<uint32_t, 4> v) {
    if constexpr (sizeof(T) == 4) {
        const vec_t<float, 4> f = __builtin_bit_cast(vec_t<float, 4>, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += f[e];
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = (e & 1) ? add_f16_mix<true>(acc[e], v[e >> 1]) : add_f16_mix<false>(acc[e], v[e >> 1]);
    }
}

// E columns from `col` of item b's output row (columns past the row left out).
template <int E>
__device__ __forceinline__ void store_slice(const SliceArgs &a, int b, int col, const float (&sum)[E]) {
    float *dst = a.out + static_cast<size_t>(b) * a.out_f + col;
    float y[E];
#pragma unroll
    for (int e = 0; e < E; ++e) y[e] = sum[e] * a.scale;
    if (a.out_vec) {
#pragma unroll
        for (int q = 0; q < E / 4; ++q)
            if (col + 4 * q < a.out_f)
                *reinterpret_cast<vec_t<float, 4> *>(dst + 4 * q) = vec_t<float, 4>{y[4 * q], y[4 * q + 1], y[4 * q + 2], y[4 * q + 3]};
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (col + e < a.out_f) dst[e] = y[e];
    }
}

// One workgroup sums one 16-byte column slice (4 f32 or 8 f16 columns) of the
// output rows of block_items items. The slice of every LUT row lies in LDS
// (stage_blocks * per tables at a time), a thread owns whole items and reads
// one 16-byte LDS row per table. LW: bytes of a staging load (16: LDS-direct
// loads; less where rows are not 16-byte aligned). IPT: items of a thread
// whose sums are held while the stages pass (1 when one stage holds every
// table; then a workgroup's later items reuse the staged slice).
// Bound by the random 16-byte LDS reads (11.7 cycles a wave read) and by the
// staging (one line request per ns and CU). With the route, against the kernel
// that gathers out of L2: 4096 items of 128 tables x 64 rows, 512 f32 columns
// 68 -> 37 us; 8192 items of 100 tables x 32 rows, 250 columns 43 -> 37 us.
// Holding a block's code words ahead spilled scalar registers: 36 us for 22.
template <typename T, int LW, int IPT>
__global__ __launch_bounds__(1024) void pairwise_gather_slice_kernel(SliceArgs a) {
    constexpr int E = kSliceBytes / static_cast<int>(sizeof(T));
    using u32x4 = vec_t<uint32_t, 4>;
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x, nthr = blockDim.x;
    // an XCD takes neighbouring slices, every item block of each: its L2 is
    // filled with those columns of the LUT only
    const int unit = xcd_block_unit(blockIdx.x, gridDim.x);
    const int slice = unit / a.nblk, blk = unit - slice * a.nblk;
    const int b_begin = blk * a.block_items, b_end = min(a.items, b_begin + a.block_items);
    if (tid < 4) reinterpret_cast<uint32_t *>(lds + a.zero_off)[tid] = 0u;

    auto stage = [&](int s) {
        const int t0 = s * a.stage_blocks * a.per, nt = min(a.stage_blocks * a.per, a.tables - t0);
        const int nrow = nt * a.rows;
        if constexpr (LW == 16) {
            const unsigned char *base = static_cast<const unsigned char *>(a.lut) +
                                        static_cast<size_t>(t0) * a.rows * a.row_bytes + slice * kSliceBytes;
            // lane l of a wave fills LDS row r0 + l; rows past the last repeat it (the LDS has room to a whole wave)
            for (int r0 = tid & ~(kWave - 1); r0 < nrow; r0 += nthr)
                __builtin_amdgcn_global_load_lds(base + static_cast<size_t>(min(r0 + (tid & (kWave - 1)), nrow - 1)) * a.row_bytes,
                                                 (__attribute__((address_space(3))) void *)(lds + __builtin_amdgcn_readfirstlane(r0) * 16),
                                                 16, 0, 0);
        } else {
            const __amdgpu_buffer_rsrc_t rsrc = buffer_rsrc(a.lut, a.lut_bytes);
            constexpr int kPieces = kSliceBytes / LW;
#pragma unroll 4
            for (int r = tid; r < nrow; r += nthr) {
                const uint32_t row = (static_cast<uint32_t>(t0) * a.rows + r) * static_cast<uint32_t>(a.row_bytes);
                vec_t<uint32_t, 4> w = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int q = 0; q < kPieces; ++q) {
                    const int off = slice * kSliceBytes + q * LW;  // a piece lies wholly inside or outside the row
                    const uint32_t voff = off < a.row_bytes ? row + off : kOutOfRange;
                    if constexpr (LW == 2) {
                        const uint32_t h = __builtin_amdgcn_raw_buffer_load_b16(rsrc, voff, 0, 0);
                        w[q >> 1] |= h << (16 * (q & 1));
                    } else if constexpr (LW == 4) {
                        w[q] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, voff, 0, 0);
                    } else {
                        const vec_t<uint32_t, 2> v =
                            __builtin_bit_cast(vec_t<uint32_t, 2>, __builtin_amdgcn_raw_buffer_load_b64(rsrc, voff, 0, 0));
                        w[2 * q] = v[0];
                        w[2 * q + 1] = v[1];
                    }
                }
                *reinterpret_cast<vec_t<uint32_t, 4> *>(lds + r * 16) = w;
            }
        }
    };

    const int rb = a.rows * kSliceBytes;  // LDS bytes of a table
    const int pass_items = nthr * IPT;
    for (int p0 = b_begin; p0 < b_end; p0 += pass_items) {
        float tot[IPT][E];
#pragma unroll
        for (int i = 0; i < IPT; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) tot[i][e] = 0.f;
        for (int s = 0; s < a.stages; ++s) {
            if (a.stages > 1 || p0 == b_begin) {  // uniform
                if (p0 != b_begin || s > 0) __syncthreads();
                stage(s);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // LDS-direct loads land before the barrier
                __syncthreads();
            }
            const int blk0 = s * a.stage_blocks, blk1 = min(a.blocks, blk0 + a.stage_blocks);
#pragma unroll 1
            for (int i = 0; i < IPT; ++i) {
                const int b = min(p0 + i * nthr + tid, b_end - 1);  // threads past the last item repeat it
                const uint32_t *wp = a.words + b;
                uint32_t w[kBlockWords];
#pragma unroll
                for (int q = 0; q < kBlockWords; ++q) w[q] = wp[static_cast<size_t>(blk0 * kBlockWords + q) * a.pitch];
                float sum[E];
#pragma unroll
                for (int e = 0; e < E; ++e) sum[e] = tot[0][e];
#pragma unroll
                for (int j = 1; j < IPT; ++j)
#pragma unroll
                    for (int e = 0; e < E; ++e) sum[e] = i == j ? tot[j][e] : sum[e];
                for (int k = blk0; k < blk1; ++k) {
                    const int n = min(a.per, a.tables - k * a.per);  // uniform
                    const int base = (k - blk0) * a.per * rb;
                    u32x4 v[kBlockTables];
                    if (n == kBlockTables) {
#pragma unroll
                        for (int u = 0; u < kBlockTables; ++u) {
                            const uint32_t code = (w[u >> 2] >> (8 * (u & 3))) & 0xFFu;
                            v[u] = *reinterpret_cast<const u32x4 *>(lds + (base + u * rb) + code * kSliceBytes);
                        }
                    } else {  // slots past the block read zeros: adding +0 changes no sum (none is -0)
#pragma unroll
                        for (int u = 0; u < kBlockTables; ++u) {
                            const uint32_t code = (w[u >> 2] >> (8 * (u & 3))) & 0xFFu;  // zero past the block
                            v[u] = *reinterpret_cast<const u32x4 *>(lds + (u < n ? base + u * rb : a.zero_off) + code * kSliceBytes);
                        }
                    }
                    // the next block's words, in flight while this one is summed
                    const int kn = min(k + 1, a.blocks - 1);
#pragma unroll
                    for (int q = 0; q < kBlockWords; ++q) w[q] = wp[static_cast<size_t>(kn * kBlockWords + q) * a.pitch];
                    float acc[E];
#pragma unroll
                    for (int e = 0; e < E; ++e) acc[e] = 0.f;
#pragma unroll
                    for (int u = 0; u < kBlockTables; ++u) add_piece<T>(acc, v[u]);
#pragma unroll
                    for (int e = 0; e < E; ++e) sum[e] = sum[e] + acc[e];
                }
#pragma unroll
                for (int j = 0; j < IPT; ++j)
#pragma unroll
                    for (int e = 0; e < E; ++e) tot[j][e] = i == j ? sum[e] : tot[j][e];
            }
        }
#pragma unroll
        for (int i = 0; i < IPT; ++i)
            if (p0 + i * nthr + tid < b_end) store_slice<E>(a, p0 + i * nthr + tid, slice * E, tot[i]);
    }
}

// ------------------------------------------------------------------ stream gather

struct StreamWordsArgs {
    const void *lut;
    const uint32_t *words;  // per = 16: word g holds tables 4 g .. 4 g + 3
    float *out;
    float scale;
    int items, out_f, tables, rows, pitch;
    int nblk;     // item blocks
    int gs;       // groups of four tables per stage
    int stages;
    int half;     // stages summed before the sums are put by (0: one run of all)
    int stagger;  // chunk pairs that do so in turn, a stage apart
};

constexpr int kStreamWThreads = 1024;
constexpr int kStreamWChunk = 64;                       // bytes of every LUT row in a workgroup's column chunk
constexpr int kStreamWSlots = kStreamWThreads / (kStreamWChunk / 16);  // 256 thread quads, IPT items each
constexpr int kStreamWBufBytes = 64 * 1024;             // a stage's LUT rows, at most (two buffers)
constexpr int kStreamWhole = 128;                       // tables summed in one run, at most
constexpr int kStreamStagger = 8;                       // a power of two

// One 16-byte LDS-direct load per lane: LDS address lds_base (wave-uniform)
// + 16 * lane. Written in assembly so that the compiler does not know that it
// writes LDS: it would make every later LDS read of either buffer wait for
// it, and the other buffer's reads are meant to overlap it. The caller waits
// for vmcnt(0) before the barrier that publishes the buffer.
__device__ __forceinline__ void lds_direct_16(const void *src, uint32_t lds_base) {
    uint32_t keep;  // m0 is given back; one wait state between its write and the load
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "s"(lds_base), "v"(src)
                 : "memory");
}

template <bool LO>
__device__ __forceinline__ float add_f16_pair(uint32_t a, uint32_t b) {  // half of a + half of b, exact products, one rounding
    float d;
    if constexpr (LO)
        asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,1]" : "=v"(d) : "v"(a), "v"(b));
    else
        asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(d) : "v"(a), "v"(b));
    return d;
}

// f16 LUTs far beyond the L2: one workgroup per (block of 256 * IPT items, 64-byte
// column chunk), the blocks of a chunk adjacent on one XCD. It walks the
// tables a stage at a time (gs groups of four, two LDS buffers, the next
// stage's rows in flight while this one is summed). In LDS the four tables of
// a group interleave, [row][table][64 bytes], so a row's address is one byte
// permute: the code over the lane's byte offset. Thread (slot, piece) owns IPT
// items and one 16-byte piece of the chunk; at a read the four slots of a
// 16-lane group take the group's four tables in turn (table k ^ (slot & 3)),
// so that their 64-byte rows fill the 256 bytes an LDS pass serves: 8 cycles
// per wave read, against 10 for rows at random and 17 when all slots read the
// same table (measured, 16-wave workgroups). A group's four rows are summed
// as (r0 + r1) + (r2 + r3), which that reordering leaves unchanged, then added
// to the item's sum. More than kStreamWhole tables are summed in two halves, the
// first half's sums lying in the output meanwhile (a second set of sums has no
// room in the registers): one run of 128 group sums is further from float64
// than the 16-table blocks of the wave-item kernel, two runs of 64 are closer
// (512 tables of 0.02 N(0, 1) 3.37e-8 in one run, 3.27e-8 in blocks, 2.97e-8 in
// halves; 128 tables 2.53e-8 every way).
// (f32 rows keep forward.hip's streamed gather, which sums
// the tables one after the other as the reference does: a sum of hundreds of
// f32 rows in another order differs from it in the last places, where f16
// rows' sums are mostly exact.)
//   1 GiB of f16 LUT (512 tables of 256 rows of 4096 columns): 4096 items 478 us
// against the wave-item kernel's 1975 us; 8192 items 815 us against the 1060 us
// of forward.hip's streamed gather (459 and 776 us in one run; the stores of the
// first half's sums are what the halves cost). The sums alone (LDS and the mixed-precision
// adds, which issue at half the rate of f32 ones) would take 2.2 us a stage
// where a stage takes 3.2 to 3.7 us.
template <int IPT>
__global__ __launch_bounds__(kStreamWThreads) void pairwise_stream_words_kernel(StreamWordsArgs a) {
    constexpr int PE = 8;  // f16 columns of a 16-byte piece
    constexpr int COLS = kStreamWChunk / 2;
    using u32x4 = vec_t<uint32_t, 4>;
    using f32x4 = vec_t<float, 4>;
    extern __shared__ __align__(16) unsigned char lds[];  // at LDS address 0: two buffers of [gs][rows][4][64] bytes, kStreamWBufBytes apart
    const int R = a.rows;
    const int unit = xcd_block_unit(blockIdx.x, gridDim.x);
    const int chunk = unit / a.nblk, blk = unit - chunk * a.nblk;
    const int tid = threadIdx.x, slot = tid >> 2, piece = tid & 3, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b0 = blk * (kStreamWSlots * IPT) + slot * IPT;
    const size_t row_bytes = static_cast<size_t>(a.out_f) * 2;
    const unsigned char *lut = static_cast<const unsigned char *>(a.lut) + static_cast<size_t>(chunk) * kStreamWChunk;
    const int gp_log2 = 31 - __builtin_clz(R) + 4;  // 16-byte pieces of a group, [row][table][piece]: R * 16

    auto issue = [&](int s, int buf) {
        const int n = a.gs << gp_log2;
        for (int i = wave * kWave; i < n; i += kStreamWThreads) {
            const int p = i + (tid & (kWave - 1));
            const int g = p >> gp_log2, q = p & ((1 << gp_log2) - 1);
            const int t = (s * a.gs + g) * 4 + ((q >> 2) & 3);
            if (p < n) {
                if (t < a.tables)
                    lds_direct_16(lut + (static_cast<size_t>(t) * R + (q >> 4)) * row_bytes + (q & 3) * 16,
                                  static_cast<uint32_t>(buf) * kStreamWBufBytes + static_cast<uint32_t>(i) * 16u);
                else  // past the last table: rows of zeros
                    *reinterpret_cast<u32x4 *>(lds + buf * kStreamWBufBytes + p * 16) = u32x4{0u, 0u, 0u, 0u};
            }
        }
    };

    // Each stage's rows are asked for once more a stage before their
    // LDS-direct loads, one word per line, the 2 * nblk workgroups that share
    // the 128-byte lines (the chunk and its neighbour, every item block) taking
    // every 2 * nblk-th row each: the loads then find the lines in L2, and HBM
    // latency does not have to fit beside one stage's sums.
    uint32_t touched = 0u;
    auto touch = [&](int s) {
        const int r = tid * 2 * a.nblk + 2 * blk + (chunk & 1), t = s * a.gs * 4 + (r >> (gp_log2 - 4));
        if (r < ((a.gs * 4) << (gp_log2 - 4)) && t < a.tables)
            touched = *reinterpret_cast<const uint32_t *>(lut + (static_cast<size_t>(s) * a.gs * 4 * R + r) * row_bytes);
    };

    // A row's LDS address: byte 0 the lane's offset in the group's interleave
    // (of table j: j * 64 + piece * 16, two tables' offsets in each of off01 and
    // off23), byte 1 the code byte (which carries the group's place in the
    // stage above the row), byte 2 the buffer.
    const uint32_t s3 = static_cast<uint32_t>(slot) & 3u;
    uint32_t off01 = (((0u ^ s3) << 6) | (piece << 4)) | ((((1u ^ s3) << 6) | (piece << 4)) << 8);
    uint32_t off23 = (((2u ^ s3) << 6) | (piece << 4)) | ((((3u ^ s3) << 6) | (piece << 4)) << 8);
    uint32_t sel[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) sel[k] = 0x0c020000u | ((4u + (k ^ s3)) << 8) | (k & 1u);
    float acc[IPT][PE];
#pragma unroll
    for (int i = 0; i < IPT; ++i)
#pragma unroll
        for (int e = 0; e < PE; ++e) acc[i][e] = 0.f;
    // IPT consecutive words of a group; slots past the pitch (a multiple of 16
    // words, the words past the last item zero) read its last IPT words, and
    // store nothing
    const uint32_t *wsrc = a.words + min(b0, a.pitch - IPT);
    constexpr int WV = IPT < 4 ? IPT : 4;  // words per load
    uint32_t w[IPT];
    auto load_words = [&](int h, const uint32_t *src) {  // words WV h .. WV h + WV - 1
        const vec_t<uint32_t, WV> v = *reinterpret_cast<const vec_t<uint32_t, WV> *>(src + WV * h);
#pragma unroll
        for (int e = 0; e < WV; ++e) w[WV * h + e] = v[e];
    };
    // the rows of tables 2 h and 2 h + 1 (in the slot's order) of item i
    auto read = [&](int i, int h, u32x4(&r)[2]) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
            r[k] = *reinterpret_cast<const __attribute__((address_space(3))) u32x4 *>(
                __builtin_amdgcn_perm(w[i], h == 0 ? off01 : off23, sel[2 * h + k]));
    };
    auto pair = [&](const u32x4(&r)[2], float(&d)[PE]) {  // their sum
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            d[2 * e] = add_f16_pair<true>(r[0][e], r[1][e]);
            d[2 * e + 1] = add_f16_pair<false>(r[0][e], r[1][e]);
        }
    };
    const int groups = (a.tables + 3) / 4;
#pragma unroll
    for (int h = 0; h < IPT / WV; ++h) load_words(h, wsrc);
    issue(0, 0);
    touch(1);
    int gi = 0;
    // the stage before which the sums are put by and the one after which they
    // are taken back: not the same for all of an XCD's chunks, or the whole
    // output would move at once
    const int turn = (chunk >> 1) & (a.stagger - 1);
    const int put = a.half != 0 ? a.half + turn : -1, get = a.half != 0 ? a.stages - 1 - turn : -1;
    // the thread's piece of its first item's output row (formed where it is
    // used: it would stay live across the sums)
    auto output = [&](int cols) {
        int t = threadIdx.x;
        __asm__ volatile("" : "+v"(t));
        return a.out + (static_cast<size_t>(blk) * (kStreamWSlots * IPT) + (t >> 2) * IPT) * a.out_f + chunk * COLS + (t & 3) * cols;
    };
    for (int s = 0; s < a.stages; ++s) {
        // this stage's rows (issued a stage ago) have landed, and every wave
        // is past its reads of the other buffer
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        asm volatile("" ::"v"(touched));
        if (s + 1 < a.stages) issue(s + 1, (s + 1) & 1);
        touch(s + 2);
        if (s == put) {  // uniform; on the way while this stage is summed
            float *to = output(4);  // (a store's four lanes fill 64 bytes)
#pragma unroll
            for (int i = 0; i < IPT; ++i, to += a.out_f) {
                if (b0 + i < a.items)
#pragma unroll
                    for (int q = 0; q < PE; q += 4)
                        *reinterpret_cast<f32x4 *>(to + 4 * q) = f32x4{acc[i][q], acc[i][q + 1], acc[i][q + 2], acc[i][q + 3]};
#pragma unroll
                for (int e = 0; e < PE; ++e) acc[i][e] = 0.f;
            }
        }
        const int g1 = min(a.gs, groups - s * a.gs);
        for (int g = 0; g < g1; ++g) {
            const uint32_t *nsrc = wsrc + static_cast<size_t>(min(++gi, groups - 1)) * a.pitch;
            // two rows are read while the two before are summed; the words of
            // the next group follow the last read of this one's
            u32x4 v0[2], v1[2];
            read(0, 0, v0);
#pragma unroll
            for (int i = 0; i < IPT; ++i) {
                float p0[PE], p1[PE];
                read(i, 1, v1);
                __builtin_amdgcn_sched_barrier(0);
                pair(v0, p0);
                if (i + 1 < IPT) read(i + 1, 0, v0);
                if ((i + 1) % WV == 0) load_words(i / WV, nsrc);
                __builtin_amdgcn_sched_barrier(0);
                pair(v1, p1);
#pragma unroll
                for (int e = 0; e < PE; ++e) acc[i][e] += p0[e] + p1[e];
            }
        }
        if (s == get) {  // uniform
            const float *from = output(4);
#pragma unroll
            for (int i = 0; i < IPT; ++i, from += a.out_f)
                if (b0 + i < a.items)
#pragma unroll
                    for (int q = 0; q < PE; q += 4) {
                        const f32x4 first = *reinterpret_cast<const f32x4 *>(from + 4 * q);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][q + e] = first[e] + acc[i][q + e];
                    }
        }
        off01 ^= 0x00010000u;
        off23 ^= 0x00010000u;
    }
    float *to = output(PE);
#pragma unroll
    for (int i = 0; i < IPT; ++i, to += a.out_f) {
        if (b0 + i < a.items) {
            float y[PE];
#pragma unroll
            for (int e = 0; e < PE; ++e) y[e] = acc[i][e] * a.scale;
            store_f32_nt<PE>(to, y);
        }
    }
}

// ------------------------------------------------------------------ host

// Kernels that address their dynamic LDS from address 0 must have no static
// LDS.
template <typename K>
bool lds_from_zero(K kernel) {
    hipFuncAttributes at{};
    return hipFuncGetAttributes(&at, reinterpret_cast<const void *>(kernel)) == hipSuccess && at.sharedSizeBytes == 0;
}

template <typename T>
hipError_t launch_slice(const SliceArgs &s, const GatherPlan &p, int lw, hipStream_t stream) {
    auto pick = [&](auto ipt) {
        constexpr int I = decltype(ipt)::value;
        if constexpr (sizeof(T) == 2)
            if (lw == 2) return pairwise_gather_slice_kernel<T, 2, I>;
        return lw == 16 ? pairwise_gather_slice_kernel<T, 16, I>
                        : lw == 8 ? pairwise_gather_slice_kernel<T, 8, I> : pairwise_gather_slice_kernel<T, 4, I>;
    };
    auto kernel = p.slice_ipt == 1 ? pick(std::integral_constant<int, 1>{}) : pick(std::integral_constant<int, kSliceIpt>{});
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), p.lds_bytes); e != hipSuccess) return e;
    return launch_kernel(TROPNN_KERNEL_FORWARD, kernel, dim3(p.wgs), dim3(p.threads), p.lds_bytes, stream, s);
}

template <int IPT>
hipError_t launch_stream_words(const StreamWordsArgs &s, const GatherPlan &p, hipStream_t stream) {
    auto kernel = pairwise_stream_words_kernel<IPT>;
    static const bool ok = lds_from_zero(kernel);
    if (!ok) return hipErrorInvalidConfiguration;
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), p.lds_bytes); e != hipSuccess) return e;
    return launch_kernel(TROPNN_KERNEL_FORWARD, kernel, dim3(p.wgs), dim3(kStreamWThreads), p.lds_bytes, stream, s);
}

hipError_t launch_stream_words_ipt(const StreamWordsArgs &s, const GatherPlan &p, hipStream_t stream) {
    switch (p.stream_ipt) {
        case 8: return launch_stream_words<8>(s, p, stream);
        case 4: return launch_stream_words<4>(s, p, stream);
        default: return launch_stream_words<2>(s, p, stream);
    }
}

// Rows off 16-byte boundaries are staged and stored in smaller pieces, which
// plan_gather's first estimate leaves out. Of those both sides are estimated
// closer, from fits to 500 shapes of 500 to 40000 items, 8 to 300 tables (the
// staged side 0.72 to 1.23 of the measured time in nine of ten). Staged although
// slower before: 346 f16 columns, 9 tables of 64 rows, 37702 items 83 us against
// 52 plain; 457 f32 columns, 46 tables of 256, 22328 items 250 against 148; 563,
// 72 of 128, 4421 items 106 against 82; 1073 f16 columns, 112 of 256, 7146 items
// 525 against 287. Kept: 619 f32 columns, 50 of 128, 37930 items 339 -> 195; 515
// f16 columns, 290 of 128, 10762 items 1102 -> 437.

// Staged: `staged` rows a workgroup slot stages in turn, in cycles of a CU
// (staged_cu) by the piece the rows' alignment leaves, more per 4-byte piece and
// less where many rows come in turn past the caches; the sums' cycles; the
// output's and the input's MB.
double slice_us(const Dims &d, int row_bytes, double staged, double staged_cu, double summed) {
    const bool f16 = d.lut_dtype == TROPNN_LUT_F16;
    double row = row_bytes % 8 == 0 ? 2.75 : row_bytes % 4 == 0 ? 3.2 : 8.1;
    if (row_bytes % 8 != 0 && staged > 16000.) row += 2.6;
    const double kcycles = 1.0 / 2400.0;  // us a cycle
    return 8.6 + kcycles * (row * staged_cu + (f16 ? 1.24 : 0.55) * summed) +
           4e-6 * d.items * (d.out_f * (d.out_f % 4 == 0 ? 0.38 : 1.23) + d.in_f * 0.19);
}

// Plain: a start, thousands of gathered elements per us and us per MB of output,
// by the lane's load (the wave-item kernel's is 16 bytes) and whether an XCD's L2
// holds the LUT.
double plain_slice_us(const Dims &d, double elements, bool in_l2) {
    struct Rate {
        double start, rate, out;
    };
    constexpr Rate kF32[3][2] = {{{6.2, 2096, 0}, {5.6, 2629, 0.29}}, {{7.9, 2731, 0}, {5.2, 2979, 0.45}}, {{11.7, 5203, 0.85}, {5.3, 7238, 1.24}}};
    constexpr Rate kF16[4][2] = {{{15.7, 2528, 0}, {9.7, 2826, 0.52}}, {{12.5, 3779, 0.13}, {7.6, 4734, 0.48}}, {{12, 3763, 0}, {12.8, 6281, 0}}, {{21.8, 10182, 0.43}, {10, 12810, 0.54}}};
    const ForwardPlan f = plan_forward(d);
    const bool f16 = d.lut_dtype == TROPNN_LUT_F16;
    const int vec = std::min(f.vec, f16 ? 4 : 2);  // (16-byte loads: rows of whole 16 bytes)
    const Rate r = f16 ? kF16[f.wave ? 3 : vec == 4 ? 2 : vec - 1][in_l2] : kF32[f.wave ? 2 : vec - 1][in_l2];
    const double us = r.start + elements / r.rate + 4e-6 * d.items * d.out_f * r.out;
    return f.wave ? 1.3 * us : us;  // (the wave-item kernel's fits are the looser ones)
}

}  // namespace

GatherPlan plan_gather(const Dims &d, bool size_only) {
    GatherPlan p{};
    const int esize = d.lut_dtype == TROPNN_LUT_F16 ? 2 : 4;
    const long long row_bytes = static_cast<long long>(d.out_f) * esize;
    const long long lut_bytes = row_bytes * d.tables * d.rows;
    if (d.items < kGatherMinItems) return p;
    // Estimated microseconds of the forward.hip kernels: gathered row elements
    // over the rates they measured, 4.2 G/us for f32 rows and 4.8 for f16; where
    // the wave-item kernel reads f16 rows 7.8, and from a LUT that an XCD's L2
    // holds 9.5 (f32 rows: 6.5); its rows that fill no power of two, f32 3.4 and
    // 4.8, f16 6 and 6.5 (1000 f16 columns, 300 tables of 64 rows, 2049 items 97 us
    // against 113 staged; 250 f32 columns, 100 tables of 32 rows, 8192 items 43
    // against 37; 800 columns, 136 tables of 64 rows, 2048 items 66 against 43)
    const double elements = 1e-3 * d.items * d.tables * d.out_f;  // thousands
    const bool wave_rows = row_bytes >= 128 && (row_bytes & (row_bytes - 1)) == 0, in_l2 = lut_bytes <= (4ll << 20);
    const bool ragged = !wave_rows && wave_tile(row_bytes) > 0;
    const double rate = ragged ? (esize == 4 ? (in_l2 ? 4800. : 3400.) : in_l2 ? 6500. : 6000.) : !wave_rows ? (esize == 4 ? 4200. : 4800.)
                                   : esize == 4 ? (in_l2 ? 6500. : 4200.) : (in_l2 ? 9500. : 7800.);
    const double plain_us = elements / rate;
    // route kernel: as many quads of items as fit 78 KB of LDS with their
    // code lists and, where they fit too, route records; at least one quad
    const int w16 = (d.tables + kBlockTables - 1) / kBlockTables;
    p.groups = w16 * kBlockWords;
    auto route_lds = [&](int quads, bool rec) {
        return static_cast<long long>(quads) * 4 * d.in_f * 4 + quads * 4ll * p.groups * 4 + (rec ? (quads * 4ll + 1) * d.tables * 8 : 0);
    };
    p.quads = 4;
    while (p.quads > 1 && route_lds(p.quads, false) > kRouteLds) p.quads >>= 1;
    p.route_rec_stage = route_lds(p.quads, true) <= kRouteLds;
    const long long rl = route_lds(p.quads, p.route_rec_stage);
    if (rl > kMaxLdsBytes) return p;  // input rows beyond a workgroup's LDS
    p.route_lds = static_cast<int>(rl);
    p.pitch = (d.items + 15) & ~15;
    p.workspace_bytes = static_cast<size_t>(p.groups) * p.pitch * sizeof(uint32_t);

    p.stream = esize == 2 && row_bytes % kStreamWChunk == 0 && d.rows >= 4 && lut_bytes >= kStreamMinLut;
    if (p.stream) {
        p.per = kBlockTables;
        const int groups = (d.tables + 3) / 4;
        p.stream_gs = kStreamWBufBytes / (d.rows * 256);
        while (p.stream_gs > 1 && p.stream_gs / 2 >= groups) p.stream_gs /= 2;  // a power of two
        if (d.tables > kStreamWhole && p.stream_gs >= groups) p.stream_gs /= 2;  // two halves, at a stage's end
        p.stream_stages = (groups + p.stream_gs - 1) / p.stream_gs;
        p.lds_bytes = kStreamWBufBytes + p.stream_gs * d.rows * 256;
        // items per thread: the least estimated time. A stage of 64 KB of rows
        // comes in 1.9 us, 2.2 us more where one item block has the rows to
        // itself, and is summed in 1.6 us and 0.26 us more per group and item
        // of a thread; one workgroup per CU, and 9 us around it (1470 shapes of
        // LUTs of 32 MiB to 1 GiB: 80 % within 10 %)
        double best = 0;
        const int chunks = static_cast<int>(row_bytes / kStreamWChunk);
        for (int ipt = 8; ipt >= 2; ipt >>= 1) {
            const int nblk = (d.items + kStreamWSlots * ipt - 1) / (kStreamWSlots * ipt);
            const long long wgs = static_cast<long long>(nblk) * chunks;
            const double stage = std::max(1.9 + 2.2 / nblk, 1.6 + 0.26 * ipt * p.stream_gs);
            const double cost = 9. + static_cast<double>((wgs + kGatherCus - 1) / kGatherCus) * p.stream_stages * stage;
            if (best == 0 || cost < best) {
                best = cost;
                p.stream_ipt = ipt;
                p.stream_nblk = nblk;
                p.wgs = static_cast<int>(wgs);
            }
        }
        // against the kernels that route and gather in one launch: thousands of
        // elements per us where the wave-item kernel or the others serve the
        // shape, by the comparisons (the fewer rows a table has, the more
        // items in flight share them). The chosen side was more than 5 % slower
        // in 24 of the 1470 shapes. 512 tables of 256 rows, us, plain against
        // staged: 128 columns, 4096 items 78 | 269, 16384 items 278 | 271; 256
        // columns 162 | 272, 630 | 298; 512 columns 239 | 216, 998 | 316; of 64
        // rows, 512 columns, 2048 items 71 | 118, 8192 items 262 | 130
        constexpr double kWaveRate[] = {13e3, 13e3, 13e3, 13e3, 13e3, 10.4e3, 7.1e3, 5.1e3, 3.7e3};
        constexpr double kItemRate[] = {6e3, 6e3, 6e3, 6e3, 6e3, 4.3e3, 3.6e3, 3.4e3, 2.9e3};
        static_assert(sizeof kWaveRate / sizeof(double) == TROPNN_MAX_COMPARISONS + 1, "one rate per comparison count");
        const ForwardPlan f = plan_forward(d);
        const double plain_rate = f.wave ? (f.wave_tile_bytes < 1024 && d.comps == 8 ? 3.3e3 : kWaveRate[d.comps]) : kItemRate[d.comps];
        p.stream_eval = best <= elements / plain_rate;
        // (training forwards that forward.hip's streamed gather would serve always
        // gain: 0.3 to 1.07 of its time at 612 of the shapes, three above 1.03)
        if (!p.stream_eval && !f.stream_ok) return p;
    } else {
        // Estimated: 15 us for two launches and the route, the staged rows at
        // one line per ns and CU (three times that in several stages, which
        // two workgroups of a CU each pass), the sums at ~12 G elements/us (16
        // with f16 rows). Measured either side of the line, plain against
        // staged: 128 f32 columns, 136 tables of 64 rows, training: 8192 items
        // 34.0 against 36.5 us, 16384 items 57 against 51 us; 512 columns, 4096
        // items 65 against 37 us; 250 columns, 100 tables of 32 rows: 2048 items
        // 19.2 against 20.2 us, 8192 items 43 against 37 us
        const double rows = static_cast<double>(d.tables) * d.rows;
        const bool one_stage = rows * kSliceBytes + 2048 <= kSliceLds;
        if (15. + 1e-3 * rows * (one_stage ? 1. : 3.) + elements / (esize == 4 ? 12000. : 16000.) > plain_us) return p;
        p.per = (d.tables + w16 - 1) / w16;
        p.blocks = (d.tables + p.per - 1) / p.per;
        p.slices = static_cast<int>((row_bytes + kSliceBytes - 1) / kSliceBytes);
        auto lds_for = [&](int sb) {
            const int rows = (std::min(sb * p.per, d.tables) * d.rows + kWave - 1) / kWave * kWave;
            return rows * kSliceBytes + 16;
        };
        // all the tables in LDS at once if they fit; else stages of at most
        // half a CU's LDS, so that one workgroup's staging overlaps
        // another's sums
        if (static_cast<long long>(d.tables) * d.rows * kSliceBytes + 2048 <= kSliceLds) {
            p.stage_blocks = p.blocks;
            p.slice_ipt = 1;
        } else {
            p.stage_blocks = 1;
            while (p.stage_blocks < p.blocks && lds_for(p.stage_blocks + 1) <= kSliceLds / 2) ++p.stage_blocks;
            p.slice_ipt = kSliceIpt;
        }
        p.stages = (p.blocks + p.stage_blocks - 1) / p.stage_blocks;
        p.lds_bytes = lds_for(p.stage_blocks);
        if (p.lds_bytes > kMaxLdsBytes) return p;
        const bool whole = row_bytes % kSliceBytes == 0;
        if (size_only && whole) {
            p.ok = true;
            return p;
        }
        p.zero_off = p.lds_bytes - 16;
        const int per_cu = p.lds_bytes > kSliceLds / 2 ? 1 : 2;
        const int max_thr = per_cu == 1 ? 1024 : 512;
        // item blocks: the least estimated time, in cycles of one CU: a
        // staged LDS row costs about one (its line's request), a wave's read
        // of 16-byte rows about 12
        double best = 0, staged = 0, summed = 0;
        const int slots = kGatherCus * per_cu;
        const int max_blk = std::max(1, std::min((d.items + kWave - 1) / kWave, 4 * slots / p.slices + 1));
        for (int nblk = 1; nblk <= max_blk;) {
            const int bi = ((d.items + nblk - 1) / nblk + kWave - 1) / kWave * kWave;
            // on to the first count of blocks with fewer items each (the cost
            // follows from bi: 524288 items of 4 columns under 200 tries of 2049)
            nblk = bi > kWave ? (d.items + bi - kWave - 1) / (bi - kWave) : max_blk + 1;
            int thr = (bi + p.slice_ipt - 1) / p.slice_ipt;
            thr = std::min(max_thr, (thr + kWave - 1) / kWave * kWave);
            if (thr < 256) thr = 256;
            const int passes = (bi + thr * p.slice_ipt - 1) / (thr * p.slice_ipt);
            const long long wgs = static_cast<long long>((d.items + bi - 1) / bi) * p.slices;
            const double stage = 1.0 * d.tables * d.rows * (p.stages > 1 ? passes : 1) + 3000.0;
            const double sum = 12.0 * passes * p.slice_ipt * (thr / kWave) * d.tables;
            const double rounds = static_cast<double>((wgs + slots - 1) / slots);
            const double cost = rounds * (stage + sum) * per_cu;
            if (best == 0 || cost < best) {
                best = cost;
                p.block_items = bi;
                p.threads = thr;
                p.wgs = static_cast<int>(wgs);
                staged = rounds * (stage - 3000.0);
                summed = rounds * sum * per_cu;
            }
        }
        // (at most 16 rows a table are staged in no time, and the fits miss those)
        if (!whole && d.rows > 16 && slice_us(d, static_cast<int>(row_bytes), staged, staged * per_cu, summed) > plain_slice_us(d, elements, in_l2)) return p;
    }
    p.ok = true;
    return p;
}

hipError_t launch_gather(const Dims &d, const GatherPlan &p, const float *x, const int64_t *anchors, const float *thr,
                         const void *lut, float scale, float *out, tropnn_route_record *rec, int64_t *indices,
                         float *margins, uint8_t *codes, uint32_t *words, hipStream_t stream) {
    const int esize = d.lut_dtype == TROPNN_LUT_F16 ? 2 : 4;
    RouteWordsArgs r{};
    r.x = x;
    r.anchors = anchors;
    r.thr = thr;
    r.words = words;
    r.rec = reinterpret_cast<uint64_t *>(rec);
    r.indices = indices;
    r.margins = margins;
    r.codes = codes;
    r.items = d.items;
    r.in_f = d.in_f;
    r.tables = d.tables;
    r.comps = d.comps;
    r.per = p.per;
    r.groups = p.groups;
    r.pitch = p.pitch;
    r.quads = p.quads;
    r.bias_mask = p.stream ? p.stream_gs - 1 : 0;
    r.table_threads = std::min(kRouteWordsThreads, (d.tables + kWave - 1) / kWave * kWave);
    r.parts = std::max(1, std::min(p.quads, kRouteWordsThreads / r.table_threads));
    r.code_off = p.quads * 4 * d.in_f * 4;
    r.rec_off = p.route_rec_stage ? r.code_off + p.quads * 4 * p.groups * 4 : 0;
    r.rec_vec = d.items % 2 == 0 && (reinterpret_cast<uintptr_t>(rec) & 15) == 0;
    const bool train = rec != nullptr, debug = indices != nullptr || margins != nullptr || codes != nullptr;
    auto route = train ? (debug ? pairwise_route_words_kernel<true, true> : pairwise_route_words_kernel<true, false>)
                       : (debug ? pairwise_route_words_kernel<false, true> : pairwise_route_words_kernel<false, false>);
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void *>(route), p.route_lds); e != hipSuccess) return e;
    const int ni = 4 * p.quads;
    if (hipError_t e = launch_kernel(TROPNN_KERNEL_FORWARD_ROUTE, route, dim3((d.items + ni - 1) / ni),
                                     dim3(r.table_threads * r.parts), p.route_lds, stream, r);
        e != hipSuccess)
        return e;
    if (p.stream) {
        StreamWordsArgs s{lut, words, out, scale, d.items, d.out_f, d.tables, d.rows, p.pitch, p.stream_nblk, p.stream_gs,
                          p.stream_stages, d.tables > kStreamWhole ? p.stream_stages / 2 : 0, p.stream_stages >= 4 * kStreamStagger ? kStreamStagger : 1};
        return launch_stream_words_ipt(s, p, stream);
    }
    SliceArgs s{};
    s.lut = lut;
    s.words = words;
    s.out = out;
    s.scale = scale;
    s.lut_bytes = static_cast<uint32_t>(static_cast<size_t>(d.tables) * d.rows * d.out_f * esize);
    s.items = d.items;
    s.out_f = d.out_f;
    s.tables = d.tables;
    s.rows = d.rows;
    s.row_bytes = d.out_f * esize;
    s.per = p.per;
    s.blocks = p.blocks;
    s.pitch = p.pitch;
    s.nblk = p.wgs / p.slices;
    s.block_items = p.block_items;
    s.stage_blocks = p.stage_blocks;
    s.stages = p.stages;
    s.zero_off = p.zero_off;
    s.out_vec = d.out_f % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    // the widest staging load that divides the rows and the LUT's address
    int lw = 16;
    while (lw > esize && ((s.row_bytes | static_cast<int>(reinterpret_cast<uintptr_t>(lut) & 15)) & (lw - 1)) != 0) lw >>= 1;
    return esize == 2 ? launch_slice<_Float16>(s, p, lw, stream) : launch_slice<float>(s, p, lw, stream);
}

}  // namespace tropnn
