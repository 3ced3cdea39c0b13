// Persistent paged GQA decode attention for query-head groups of 1 to 16 heads, unit dim
// stride -- the pipelined MFMA kernel.
//
// What bounds it: the K/V rows are read once, so the chip's rate of scattered 256 B row reads
// does (6.1 TB/s measured for a plain gather of the 395 MB of a 64-request 8B-class layer's rows, 6.4
// with the rows of one head after the other, 6.6 streaming as many bytes in one launch) -- as long as
// enough of them are in flight.  A worker that stops loading at a task's end (merge barrier, then claim ->
// record -> indices -> rows, a round trip each) leaves its share unused, and so does a wave
// whose tile math takes as long as the rows' round trip.  Hence:
//
// * The math runs on the matrix cores, also for small groups: a 16 KB tile takes 16 (group <= 16)
//   MFMAs and 325 (8 heads) to 340 (4 heads) VALU instructions, all of a launch's counted, against ~790
//   for packed dot products with 4 heads.
// * Loads cross task boundaries.  A helper wave beside the kWaves compute waves finds the
//   worker's next task while the current one streams, and leaves its record, its q rows
//   and the first tiles' indices in LDS (two slots by task parity).  A compute wave
//   that runs out of tiles requests its first tile of the next task before it hands over its
//   share of the merge, and the merge's own LDS rows alternate by task parity, so a task
//   costs one workgroup barrier, crossed with loads in flight.
// * Rows are fetched whole, 16 lanes of 16 B.  The MFMA's own operand layout (64 B of 16 rows an
//   instruction) moves the same bytes slower: 78.9 against 71.6 us for the layer named below,
//   both in an eight-wave form.  So K rows pass through a wave's LDS tile; V rows are
//   operands as they come.
//
// Measured, us a layer of a captured step with its plan and merges (before = a VALU kernel for groups up
// to 4 and a separate MFMA kernel with 64 B row pieces): 8B-class heads, 64 requests, 395 MB 81.3 -> 79.9
// (the kernel alone 72.6); 70B-class heads, 32 requests in 16-token pages, 1.14 GB 211.7 -> 203.4; 32 kv
// heads, no grouping, 537 MB 112.0 -> 103.5; head_dim 64 65.6 -> 58.3; head_dim 256 91.8 -> 85.8; one request
// of 8k tokens 21.6 -> 17.0; one kv head of 8 query heads, 64 requests 28.7 -> 24.9.
//
// Lane l of a compute wave is (m, j) = (l % 16, l / 16).  MFMA operands of 16x16xK:
// A[m][kj ..], B[kj ..][n = l % 16], D[4j + i][n], each lane group j holding K / 4
// consecutive k.  One tile of a (record, kv head), kTile tokens:
//   S^T = K . Q^T    M = 16 tokens, N = 16 heads (lane columns past the group repeat its
//                    heads and are not stored), contraction D in 32-dim chunks; K (A) comes from the
//                    staged tile, the q rows (B) from LDS.  Lane (n, j) gets head n's scores of
//                    tokens 16h + 4j + i.
//   softmax          per head, exp2 domain, fp32; the cross-lane maximum and the rescaling only in
//                    tiles that raise some head's maximum.  (Letting scores exceed the maximum
//                    by 2^8 first is no faster, and the largest p is then not the 1 that rounds
//                    exactly: 2.2e-3 instead of 1.75e-3 off in bf16 without remainders, 1.66e-3 of it
//                    the result's own rounding.)  P is rounded to the KV dtype (kernels/attention.py:78), and where
//                    fewer waves share a task than would keep that error down its remainder
//                    is multiplied too (below).
//   O^T += V^T . P^T the B operand is P as S^T left it; the A operand needs one dim of each of
//                    the lane group's tokens per lane: lane (m, j) loads kRowDims consecutive dims
//                    of each of its tokens and block b takes element b (v_perm), so output row r
//                    of block b is dim kRowDims r + b (D = 256: 128 h + 8 r + b).
// The next tile's rows are requested into the registers this tile's free up, V after P.V.
//
// The remainder of P: a wave's largest p is 1 and rounds exactly, the other p of the heavy tokens do
// not, so the fewer waves share a task the larger the error of the rounded P: against 64 bits, in bf16
// before the output's rounding, 4.6e-4 with eight waves (groups up to 4 in an earlier kernel), 5.8e-4
// with four, 6.2e-4 with three.  So groups up to 4, and head_dim 256 (three waves), multiply
// P - round(P) in the KV dtype as well, which leaves 1e-6.  Groups up to 4 leave the MFMA's upper 8
// columns free: column n + 8 takes the remainders of head n, at no MFMA more, and they go to merge rows
// of their own (added in registers at the task's end: 0.6 to 1.1 us a launch more).  8 and 16 heads at
// D = 256, which have no LDS for such rows, take a second MFMA a block into accumulators of their own.
// It costs up to 2 % of a layer's time for groups up to 4 (eight layers of 64 requests 637.5 -> 638.9 us,
// 16 of one request 269 -> 272.5; 4 % with 128 requests of ~60 tokens, 20.4 -> 21.2), 1 to 8 % for the
// others (48 requests of ~1000 tokens, D 256: 8 heads 86.1 -> 87.6, 16 heads 60.9 -> 63.4).
//
// Geometry: two workgroups must be resident per CU (the default worker count), and the hardware
// deals a workgroup's waves to the SIMDs in turn, so five waves take two slots of one SIMD:
// 4 + 1 waves need 128 VGPRs (at 140 only every second workgroup starts), as do 7 + 1 at D = 64;
// at D = 256, where a tile and its output are 128 registers, 3 + 1 waves have 256.  (The paged builds of
// 8 and 16 heads at D = 128, and those of pages that are no power of two, spill one or two VGPRs: a
// store where a wave starts and a load in its helper, none in a loop.)  At 16 tokens a tile D = 128
// fits 8 + 1 waves only with spills: 75 us for the first layer above.  64-token tiles at D = 64 (4 + 1
// waves): 57.0 against 52.9 us.
#include <float.h>

#include "valu_ops.h"

namespace sgd {
namespace {

using valu::uni;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr int kIndptrLds = 256;   // CSR: kv_indptr entries kept in LDS (rows beyond read memory)
// Tiles of wave 0 left when the helper claims the next unit: the search takes about three tiles'
// time.  1 / 2 / 3 / 5: 78.0 / 77.3 / 79.0 / 79.4 us a layer (64 requests; runs of one differ by up to 2.0),
// 191 / 193 / 199 / 200 (70B class; by up to 5.8), the others within 1 of each other: it hardly matters.
constexpr int kClaimLead = 3;
constexpr int kOPad = 4;          // floats after a merge row: its 16 B stores spread over the banks
constexpr int kQPad = 16;         // bytes after a q row: 16 heads' 16 B reads spread over the banks

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int D>
struct PGeo {
    static_assert(D == 64 || D == 128 || D == 256, "head_dim 64, 128 or 256");
    static constexpr int kWaves = D == 64 ? 7 : D == 128 ? 4 : 3;  // compute waves per workgroup
    static constexpr int kThreads = 64 * (kWaves + 1);
    // The next K rows are requested once this tile's are staged, or not beside the scores and their
    // operands but after them: at D = 128 for want of registers, at D = 256, which has them, because the
    // early request is no faster (24 requests 86.1 us a layer against 85.6, others -1 to +2 %).
    static constexpr bool kEarlyK = D == 64;
    static constexpr int kWavesPerSimd = D == 256 ? 2 : 4;
    static constexpr int kTile = D == 256 ? 16 : 32; // tokens per tile
    static constexpr int kHalves = kTile / 16;       // 16-token blocks of S^T
    static constexpr int kChunks = D / 32;           // QK contraction chunks
    static constexpr int kVals = kTile / 4;          // tokens per lane: scores, P values, V slots
    static constexpr int kVWords = D / 32;           // 32-bit words of V per lane and slot
    static constexpr int kBlocks = D / 16;           // O^T blocks
    static constexpr int kRowDims = D == 64 ? 4 : 8; // dims per output row: row r of block b is dim kRowDims r + b
    static constexpr int kKLoads = kTile * D / 512;  // 16 B loads per lane for a tile's K rows
    static constexpr int kStage = kTile * 2 * D;     // bytes of a wave's K tile in LDS
    static constexpr int kQRow = 2 * D + kQPad;      // bytes of a q row in LDS
    static constexpr int kORow = D + kOPad;          // floats of a merge row in LDS
};

// A task as the helper publishes it; task < 0 ends the worker's stream.
struct Slot {
    int32_t task, request, split, start, end, group, ind0, pad;
};

template <int D>
struct PipeShared {
    char kstage[PGeo<D>::kWaves][PGeo<D>::kStage];  // per wave: the tile's K rows (k_pos)
    Slot slot[2];
    int32_t seq[2];   // k + 1 once slot k & 1 holds task k of this worker
    int32_t started;  // tiles that wave 0 has started since the launch
    int32_t pad;
    int32_t idx[2][PGeo<D>::kTile * PGeo<D>::kWaves];  // page/slot indices of the first kWaves tiles
    float m[2][PGeo<D>::kWaves][16], d[2][PGeo<D>::kWaves][16];
    int32_t indptr[kIndptrLds];
    // then q rows [2][G][kQRow bytes] and merge rows [merge_sets(G)][kWaves][merge_heads(G)][kORow]
};

// The merge rows share a CU's 160 KB with a second workgroup: two sets, alternating by task
// parity (one barrier per task), where they fit, else one set and a second barrier; 16 heads
// at D = 256 are merged in two passes over one set (67 KB; 123 requests of ~100 tokens, 16 heads a
// group: 53.9 us, 61.0 in four passes of half the rows).
template <int D>
__host__ __device__ constexpr int pass_heads(int g) { return D == 256 && g > 8 ? 8 : g; }
template <int D>
__host__ __device__ constexpr int merge_sets(int g) { return g <= (D == 256 ? 4 : 8) ? 2 : 1; }

// Workgroup barriers that end a task.
template <int D>
__host__ __device__ constexpr int merge_barriers(int g) { return merge_sets<D>(g) == 2 ? 1 : 2 * (g / pass_heads<D>(g)); }

// How a task's remainders of P are multiplied (above).
enum Rest { kNoRest, kRestColumns, kRestOwn };
template <int D>
__host__ __device__ constexpr Rest rest_form(int g) { return g <= 4 ? kRestColumns : D == 256 ? kRestOwn : kNoRest; }

// Rows of a wave's share of the merge: those of the remainders after the heads'.
template <int D>
__host__ __device__ constexpr int merge_heads(int g) {
    return rest_form<D>(g) == kRestColumns ? 2 * g : pass_heads<D>(g);
}

template <int D>
__host__ __device__ constexpr int pipe_lds_bytes(int g) {
    return (int)sizeof(PipeShared<D>) + 2 * g * PGeo<D>::kQRow +
           merge_sets<D>(g) * PGeo<D>::kWaves * merge_heads<D>(g) * PGeo<D>::kORow * (int)sizeof(float);
}
template <int D>
constexpr bool two_per_cu() {
    for (int g = 1; g <= 16; g *= 2)
        if (pipe_lds_bytes<D>(g) > 80 * 1024) return false;
    return true;
}
static_assert(two_per_cu<64>() && two_per_cu<128>() && two_per_cu<256>(), "two workgroups per CU");

template <int DT>
__device__ __forceinline__ f32x4 mfma32(uint4 a, uint4 b, f32x4 c) {
    if constexpr (DT == SGD_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
}

template <int DT>
__device__ __forceinline__ f32x4 mfma16(uint2 a, uint2 b, f32x4 c) {
    if constexpr (DT == SGD_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a), __builtin_bit_cast(i16x4, b),
                                                          c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0,
                                                      0, 0);
}

// Row loads from an address computed in integers: named as global memory, or they would be
// flat loads, which count as LDS accesses too and are waited for all at once.
__device__ __forceinline__ uint4 load_row16(uint64_t p) {
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    typedef const __attribute__((address_space(1))) v4u gv4u;
    const v4u t = __builtin_nontemporal_load((gv4u *)p);
    return make_uint4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ uint2 load_row8(uint64_t p) {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(1))) v2u gv2u;
    const v2u t = __builtin_nontemporal_load((gv2u *)p);
    return make_uint2(t.x, t.y);
}

// Token (within the tile) of V slot s of lane group j: that of S^T value s of the lane.
__device__ __forceinline__ int slot_token(int j, int s) { return 16 * (s >> 2) + 4 * j + (s & 3); }

// Uniform: where a wave's next tile comes from.
struct Source {
    const char *kbase, *vbase;  // K / V + kv head (bytes)
    const int32_t *rows;        // the request's page table row / kv_indices
    int32_t tok, end;           // first token of the tile, end of the task
};

template <int D>
struct TileRegs {
    uint4 k[PGeo<D>::kKLoads];
    uint32_t v[PGeo<D>::kVals][PGeo<D>::kVWords];
    int32_t idx[PGeo<D>::kHalves];  // index of token 16h + 4j + m % 4 of the tile to request next
};

// Row and 16 B piece that lane (m, j) fetches with K load i: whole 256 B (D = 64: 128 B) rows per
// 16 (8) lanes, four (eight) rows an instruction, and not the MFMA's operand layout itself, 64 B of 16
// rows an instruction (at the top: 78.9 against 71.6 us), so the rows pass through LDS.
template <int D>
__device__ __forceinline__ int k_row(int i, int m, int j) {
    if constexpr (D == 64) return 16 * (i >> 1) + 4 * j + 2 * (i & 1) + (m >> 3);
    else if constexpr (D == 128) return 16 * (i >> 2) + 4 * j + (i & 3);
    else return 4 * j + (i & 3);
}
template <int D>
__device__ __forceinline__ int k_piece(int i, int m) {
    if constexpr (D == 64) return m & 7;
    else if constexpr (D == 128) return m;
    else return 16 * (i >> 2) + m;
}

// Byte position of piece c of row t in a staged K tile.  The XOR spreads the 16 rows that a 16 B
// read takes at once over all 64 banks (rows are 128, 256 or 512 B).  Both uses split it into
// a position per lane and an XOR and offset per load, so that one register serves all.
template <int D>
__device__ __forceinline__ constexpr int k_swizzle(int t) { return D == 64 ? (t >> 1) & 7 : t & 15; }

// Where the lane's K load i goes: k_pos(k_row(i), k_piece(i)) from its position for load 0.
template <int D>
__device__ __forceinline__ int k_write_pos0(int m, int j) {
    const int t = k_row<D>(0, m, j);
    return t * 2 * D + ((k_piece<D>(0, m) ^ k_swizzle<D>(t)) << 4);
}
template <int D>
__device__ __forceinline__ int k_write_pos(int pos0, int i) {
    // rows: +1 per load (D = 64: +2 for odd loads, +16 per pair); pieces: +16 per four loads at D = 256
    if constexpr (D == 64) return (pos0 ^ ((i & 1) << 4)) + (i & 1) * 256 + (i >> 1) * 2048;
    else return (pos0 ^ ((i & 3) << 4)) + (i & 3) * 2 * D + (i >> 2) * (D == 128 ? 16 * 256 : 256);
}
// Where the lane reads row 16h + m's dims 32c + 8j .. +7 (piece 4c + j).
template <int D>
__device__ __forceinline__ int k_read_pos0(int m, int j) { return m * 2 * D + ((j ^ k_swizzle<D>(m)) << 4); }
template <int D>
__device__ __forceinline__ int k_read_pos(int pos0, int h, int c) {
    // D = 256 pieces 16 .. 31 (c >= 4) lie 256 B further, outside the swizzled bits
    return (pos0 ^ ((c & 3) << 6)) + (c >> 2) * 256 + h * 16 * 2 * D;
}

// Where dim d of an output lies in a merge row: a lane's O^T block (rows 4j .. 4j + 3) is stored
// as it stands, 16 B.
template <int D>
__device__ __forceinline__ constexpr int merge_pos(int d) {
    constexpr int n = PGeo<D>::kRowDims;
    return (d & ~(4 * n - 1)) + 4 * (d % n) + (d / n) % 4;
}

// Indices of the tile at tok; tokens past the end repeat the last one, so every address is
// in bounds and the loads need no branch.
template <bool CSR, int D, bool kPow2>
__device__ __forceinline__ void load_indices(const sgd_decode_args &a, const Source &s, int32_t tok,
                                             const PageMap<kPow2> &pm, int lane, TileRegs<D> &r) {
    const int m = lane & 15, j = lane >> 4;
#pragma unroll
    for (int h = 0; h < PGeo<D>::kHalves; ++h) {
        const int32_t t = min(tok + 16 * h + 4 * j + (m & 3), s.end - 1);
        r.idx[h] = CSR ? s.rows[t] : s.rows[(int64_t)pm.page(t) * a.pt_stride[1]];
    }
}

// Address in K or V (kv head at `base`) of token 16h + 4j + m % 4 of the tile at s, from its index.
template <bool CSR, bool kPow2>
__device__ __forceinline__ uint64_t row_address(const char *base, int32_t idx, int h, const Source &s,
                                                const PageMap<kPow2> &pm, int lane, const int64_t (&stride)[4]) {
    int64_t step = stride[0] * 2;
    asm volatile("" : "+s"(step));  // bytes before the product, not after
    uint64_t p = reinterpret_cast<uintptr_t>(base) + (uint64_t)(uint32_t)idx * step;
    if constexpr (!CSR) {
        const int32_t t = min(s.tok + 16 * h + 4 * (lane >> 4) + (lane & 3), s.end - 1);
        p += (int64_t)(uint32_t)pm.row(t) * (stride[1] * 2);
    }
    return p;
}

// Byte `col` of the row of token 16h + 4j + I, whose address lane 4 (..) + I of each group holds.
template <int I>
__device__ __forceinline__ uint64_t token_row(uint64_t p, uint32_t col) {  // quad_perm [I, I, I, I]
    typedef uint32_t v2u __attribute__((ext_vector_type(2)));
    const v2u w = __builtin_bit_cast(v2u, p);
    const v2u r = {(uint32_t)valu::dpp_i<0x55 * I>((int32_t)w.x), (uint32_t)valu::dpp_i<0x55 * I>((int32_t)w.y)};
    return __builtin_bit_cast(uint64_t, r) + col;
}

template <bool CSR, int D, bool kPow2>
__device__ __forceinline__ void issue_k(const sgd_decode_args &a, const Source &s, const PageMap<kPow2> &pm, int lane,
                                        TileRegs<D> &r) {
    using G = PGeo<D>;
    const int m = lane & 15;
    const uint32_t col = 16 * k_piece<D>(0, m);
    // 16 tokens at a time: their addresses are in registers together
#pragma unroll
    for (int h = 0; h < G::kHalves; ++h) {
        const uint64_t p = row_address<CSR>(s.kbase, r.idx[h], h, s, pm, lane, a.k_stride);
        if constexpr (D == 64) {
            auto row = [&](uint64_t lo, uint64_t hi) { return m & 8 ? hi : lo; };
            r.k[2 * h] = load_row16(row(token_row<0>(p, col), token_row<1>(p, col)));
            r.k[2 * h + 1] = load_row16(row(token_row<2>(p, col), token_row<3>(p, col)));
        } else {
#pragma unroll
            for (int w = 0; w < D / 128; ++w) {  // 256 B of the rows at a time
                r.k[4 * (h + w)] = load_row16(token_row<0>(p, col) + 256 * w);
                r.k[4 * (h + w) + 1] = load_row16(token_row<1>(p, col) + 256 * w);
                r.k[4 * (h + w) + 2] = load_row16(token_row<2>(p, col) + 256 * w);
                r.k[4 * (h + w) + 3] = load_row16(token_row<3>(p, col) + 256 * w);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The V rows of the tile at s, and the indices of the wave's tile after it.  The index loads go
// out between the V addresses, which use up the old indices, and the V loads: in the order K,
// indices, V the wait for the next K addresses leaves V in flight (the counter of
// outstanding loads counts in order).
template <bool CSR, int D, bool kPow2>
__device__ __forceinline__ void issue_v(const sgd_decode_args &a, const Source &s, const PageMap<kPow2> &pm, int lane,
                                        TileRegs<D> &r) {
    using G = PGeo<D>;
    const uint32_t col = (D == 64 ? 8 : 16) * (lane & 15);
    uint64_t p[G::kHalves];
#pragma unroll
    for (int h = 0; h < G::kHalves; ++h) p[h] = row_address<CSR>(s.vbase, r.idx[h], h, s, pm, lane, a.v_stride);
    __builtin_amdgcn_sched_barrier(0);
    load_indices<CSR, D>(a, s, s.tok + G::kTile * G::kWaves, pm, lane, r);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < G::kHalves; ++h) {
        const uint64_t row[4] = {token_row<0>(p[h], col), token_row<1>(p[h], col), token_row<2>(p[h], col),
                                 token_row<3>(p[h], col)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t(&w)[G::kVWords] = r.v[4 * h + i];
            if constexpr (D == 64) {
                const uint2 t = load_row8(row[i]);
                w[0] = t.x, w[1] = t.y;
            } else {
#pragma unroll
                for (int hv = 0; hv < D / 128; ++hv) {
                    const uint4 t = load_row16(row[i] + 256 * hv);
                    w[4 * hv] = t.x, w[4 * hv + 1] = t.y, w[4 * hv + 2] = t.z, w[4 * hv + 3] = t.w;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// A wave's softmax state and output: lane (n, j) holds head n's maximum and its own tokens'
// share of the denominator, and dims of rows 4j + i of each O^T block (kRestOwn: of the remainders too).
template <int D, Rest kRest>
struct State {
    float m, den;
    f32x4 o[PGeo<D>::kBlocks];
    f32x4 rest[kRest == kRestOwn ? PGeo<D>::kBlocks : 1];
};

// a - its value in the KV dtype, for both halves of a packed pair; where `keep` is 0 the pair itself.
template <int DT>
__device__ __forceinline__ uint32_t remainder2(uint32_t w, float lo, float hi, uint32_t keep) {
    w &= keep;
    return valu::pack2<DT>(lo - to_f32<DT>(w & 0xffff), hi - to_f32<DT>(w >> 16));
}

// The remainders' share of an output, to add to that of the rounded P.  An infinite V row makes the latter
// infinite, which 0 x infinity or an infinity of the other sign here must not turn into NaN.
__device__ __forceinline__ float finite(float rest) { return __builtin_amdgcn_fmed3f(rest, -FLT_MAX, FLT_MAX); }

// One tile of nvalid tokens, whose rows are in (or on their way to) r; the tile at `s` is
// requested into the same registers as they become free.
template <int DT, bool CSR, int D, bool kPow2, Rest kRest>
__device__ __forceinline__ void tile_step(const sgd_decode_args &a, TileRegs<D> &r, char *stage, const char *q,
                                          int32_t nvalid, float scale2, const Source &s, const PageMap<kPow2> &pm,
                                          int lane, State<D, kRest> &st) {
    using G = PGeo<D>;
    constexpr int kV = G::kVals;
    // per-lane positions are rebuilt each tile, not held live
    asm volatile("" : "+v"(lane));
    const int m = lane & 15, j = lane >> 4;
    const int wpos = k_write_pos0<D>(m, j), rpos = k_read_pos0<D>(m, j);
#pragma unroll
    for (int i = 0; i < G::kKLoads; ++i) *reinterpret_cast<uint4 *>(stage + k_write_pos<D>(wpos, i)) = r.k[i];
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (G::kEarlyK) issue_k<CSR, D>(a, s, pm, lane, r);
    wave_sync();
    __builtin_amdgcn_sched_barrier(0);
    f32x4 sc[G::kHalves];
#pragma unroll
    for (int h = 0; h < G::kHalves; ++h) sc[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < G::kChunks; ++c) {
        const uint4 qc = *reinterpret_cast<const uint4 *>(q + 64 * c);
#pragma unroll
        for (int h = 0; h < G::kHalves; ++h)
            sc[h] = mfma32<DT>(*reinterpret_cast<const uint4 *>(stage + k_read_pos<D>(rpos, h, c)), qc, sc[h]);
        // operands of one chunk at a time in registers (D = 128 has room for two)
        __builtin_amdgcn_sched_barrier(0);
    }
    wave_sync();  // the next tile's rows overwrite these
    float x[kV];
#pragma unroll
    for (int i = 0; i < kV; ++i) x[i] = sc[i >> 2][i & 3] * scale2;
    if (nvalid < G::kTile) {  // rows past the task's end: no score, and zero V (their p is exactly zero)
#pragma unroll
        for (int i = 0; i < kV; ++i) {
            const bool off = slot_token(j, i) >= nvalid;
            x[i] = off ? -INFINITY : x[i];
#pragma unroll
            for (int w = 0; w < G::kVWords; ++w) r.v[i][w] = off ? 0u : r.v[i][w];
        }
    }
    float mx = x[0];
#pragma unroll
    for (int i = 1; i < kV; ++i) mx = fmaxf(mx, x[i]);
    if (__ballot(mx > st.m) != 0) {
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(st.m, mx);
        const float alpha = __builtin_amdgcn_exp2f(st.m - m_new);
        st.m = m_new;
        st.den *= alpha;
#pragma unroll
        for (int b = 0; b < G::kBlocks; ++b) {
            st.o[b] = st.o[b] * alpha;
            if constexpr (kRest == kRestOwn) st.rest[b] = st.rest[b] * alpha;
        }
    }
    float p[kV];
#pragma unroll
    for (int i = 0; i < kV; ++i) {
        p[i] = __builtin_amdgcn_exp2f(x[i] - st.m);
        st.den += p[i];
    }
    uint32_t pw[kV / 2];  // P in the KV dtype, token pairs
#pragma unroll
    for (int i = 0; i < kV; i += 2) pw[i / 2] = valu::pack2<DT>(p[i], p[i + 1]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!G::kEarlyK) issue_k<CSR, D>(a, s, pm, lane, r);
    __builtin_amdgcn_sched_barrier(0);
    // The remainders, behind the request of the next K rows, whose round trip a wave's next tile waits for
    // (before it: 90.4 us for 32 mixed requests of 16-token pages, plan and merge included; 88.3 here).
    uint32_t rest[kRest == kRestOwn ? kV / 2 : 1];
    if constexpr (kRest == kRestOwn) {
#pragma unroll
        for (int i = 0; i < kV; i += 2) rest[i / 2] = remainder2<DT>(pw[i / 2], p[i], p[i + 1], 0xffffffffu);
    } else if constexpr (kRest == kRestColumns) {
        const uint32_t keep = m & 8 ? 0xffffffffu : 0u;
#pragma unroll
        for (int i = 0; i < kV; i += 2) pw[i / 2] = remainder2<DT>(pw[i / 2], p[i], p[i + 1], keep);
    }
    // 32 tokens per MFMA; the 16 of a D = 256 tile take the K = 16 one
#pragma unroll
    for (int t = 0; t < kV; t += 8) {
        const uint32_t *pk = pw + t / 2;
#pragma unroll
        for (int b = 0; b < G::kBlocks; ++b) {
            const uint32_t sel = (b & 1) ? 0x07060302u : 0x05040100u;
            auto pair = [&](int i) { return __builtin_amdgcn_perm(r.v[t + i + 1][b >> 1], r.v[t + i][b >> 1], sel); };
            if constexpr (kV >= 8) {
                static_assert(kV < 8 || kRest != kRestOwn, "remainders in a second MFMA: the 16-token tile's");
                st.o[b] = mfma32<DT>(make_uint4(pair(0), pair(2), pair(4), pair(6)),
                                     make_uint4(pk[0], pk[1], pk[2], pk[3]), st.o[b]);
            } else {
                const uint2 v = make_uint2(pair(0), pair(2));
                st.o[b] = mfma16<DT>(v, make_uint2(pk[0], pk[1]), st.o[b]);
                if constexpr (kRest == kRestOwn) st.rest[b] = mfma16<DT>(v, make_uint2(rest[0], rest[1]), st.rest[b]);
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    issue_v<CSR, D>(a, s, pm, lane, r);
    __builtin_amdgcn_sched_barrier(0);
}

// Tiles of a task that wave `wave` computes (tile t -> wave t % kWaves).
template <int D>
__device__ __forceinline__ int32_t wave_tiles(int32_t start, int32_t end, int wave) {
    constexpr int kTile = PGeo<D>::kTile, kWaves = PGeo<D>::kWaves;
    const int32_t n = (int32_t)((uint32_t)(max(end - start, 0) + kTile - 1) / kTile);  // none for end < start
    return n > wave ? (int32_t)((uint32_t)(n - wave + kWaves - 1) / kWaves) : 0;
}

// ------------------------------------------------------------------ helper wave
// Walks the worker's units (a task in R0, R1 and STATIC, a pack in D1/D4; modes and claims as
// in for_each_task of attention_common.h) one task ahead of the compute waves.
template <bool CSR, int D, bool kPow2>
__device__ __forceinline__ void helper_wave(const sgd_decode_args &a, PipeShared<D> &sh, char *sq, int32_t G, int lane,
                                            const PageMap<kPow2> &pm) {
    using GG = PGeo<D>;
    // The launch's scalars and the worker's first entry in one round trip: in every mode but
    // R0 and STATIC the first unit is the worker's own index.
    const int32_t worker = blockIdx.x;
    if (lane == 0) {  // LDS holds an earlier workgroup's values; seq[0] is written before the first barrier
        sh.seq[1] = 0;
        sh.started = 0;
    }
    const bool table = a.dispatch != nullptr;
    const bool early = table && worker < a.dispatch_units;
    Entry e{};
    if (early) e = load_entry(a.dispatch, worker);
    const int32_t mode_v = *a.mode, records_v = *a.record_count, packs_v = a.num_packs ? *a.num_packs : 0;
    const int32_t rows_v = CSR && a.active ? *a.active + 1 : 0;
    const int32_t mode = uni(mode_v), total = uni(records_v) * a.kv_heads;
    const bool dynamic = mode >= 3;
    const int32_t limit = dynamic ? uni(packs_v) : total;
    const int32_t iptr_n = CSR ? min(uni(rows_v), kIndptrLds) : 0;
    bool iptr_ready = false;

    int32_t first = 0, count = 0, i = 0, after = -1;
    TaskInfo info{};
    // Opens `unit`: its first task's record in `info`; false past the last unit.
    auto open = [&](int32_t unit, bool have) {
        if (unit < 0 || unit >= limit) return false;
        if (!have) {
            have = table && mode != 0 && unit < a.dispatch_units;
            if (have) e = load_entry(a.dispatch, unit);
        }
        const Unit u = unit_of(a, unit, mode, have, e);
        first = u.first;
        count = u.count;
        i = 0;
        after = dynamic ? -1 : mode == 2 ? uni(a.static_next[unit]) : unit + a.workers;
        info = uniform_info(u.resolved ? u.info : decode_task(a, first, mode));
        return true;
    };
    bool live = open(mode == 2 ? uni(a.static_head[worker]) : worker, early && mode != 0 && mode != 2);
    int32_t wave0_tiles = 0;  // wave 0's tiles of the tasks before task k

    for (int32_t k = 0;; ++k) {
        // ---- publish task k (read last before the barrier that ended task k - 2)
        Slot &slot = sh.slot[k & 1];
        if (live) {
            const int32_t ind0 = !CSR ? 0
                                 : iptr_ready && info.request < iptr_n ? uni(sh.indptr[info.request])
                                                                       : uni(a.indptr[info.request]);
            const int32_t *rows = CSR ? a.pages + ind0 : a.pages + (int64_t)info.request * a.pt_stride[0];
            // A record without a token has no last one to repeat (end - 1 may lie before the table), and
            // nothing uses its indices: it reads its request's first page, or kv_indptr's first word.  (A
            // branch spills up to 47 SGPRs more, another word's pointer 37: 0.6 us a launch of one request.)
            const bool some = info.end > info.start;
            if constexpr (CSR) rows = some ? rows : a.indptr;
            const int32_t last = some ? info.end - 1 : 0;
            constexpr int kIdx = GG::kTile * GG::kWaves, kLoads = (kIdx + 63) / 64;
            int32_t tile_idx[kLoads];
#pragma unroll
            for (int t = 0; t < kLoads; ++t) {
                const int32_t tok = min(info.start + 64 * t + lane, last);
                tile_idx[t] = CSR ? rows[tok] : rows[(int64_t)pm.page(tok) * a.pt_stride[1]];
            }
            // the group's q rows, 16 B pieces (head = piece / (D / 8))
            char *dst = sq + (k & 1) * G * GG::kQRow;
            const uint16_t *qp = static_cast<const uint16_t *>(a.q) + (int64_t)info.request * a.q_stride[0] +
                                 (int64_t)info.group * G * a.q_stride[1];
            const int64_t qd = a.q_stride[2];
            for (int32_t c = lane; c < G * (D / 8); c += 64) {
                const int32_t h = c / (D / 8), d8 = c % (D / 8);
                const uint16_t *p = qp + h * a.q_stride[1] + d8 * 8 * qd;
                uint4 w;
                if (qd == 1 && (reinterpret_cast<uintptr_t>(p) & 15) == 0) {
                    w = *reinterpret_cast<const uint4 *>(p);
                } else {
                    uint32_t w4[4] = {0, 0, 0, 0};
#pragma unroll
                    for (int x = 0; x < 8; ++x) w4[x >> 1] |= (uint32_t)p[x * qd] << (16 * (x & 1));
                    w = make_uint4(w4[0], w4[1], w4[2], w4[3]);
                }
                *reinterpret_cast<uint4 *>(dst + h * GG::kQRow + d8 * 16) = w;
            }
#pragma unroll
            for (int t = 0; t < kLoads; ++t)
                if (64 * t + lane < kIdx) sh.idx[k & 1][64 * t + lane] = tile_idx[t];
            if (lane == 0) slot = Slot{first + i, info.request, info.split, info.start, info.end, info.group, ind0, 0};
        } else if (lane == 0) {
            slot.task = -1;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        if (lane == 0) __hip_atomic_store(&sh.seq[k & 1], k + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (k > 0)
            for (int b = merge_barriers<D>(G); b > 1; --b) lds_barrier();
        lds_barrier();  // task k - 1 ends (k = 0: the stream starts)
        if (!live) break;

        // ---- find task k + 1
        if constexpr (CSR) {
            if (!iptr_ready) {
                for (int t = lane; t < iptr_n; t += 64) sh.indptr[t] = a.indptr[t];
                wave_sync();
                iptr_ready = true;
            }
        }
        const int32_t n0 = wave_tiles<D>(info.start, info.end, 0);
        if (i + 1 < count) {
            ++i;
            const int32_t task = first + i;
            if (task % a.kv_heads != 0) ++info.group;  // the same record's next head
            else info = uniform_info(decode_task(a, task, mode));
        } else if (dynamic) {
            // not before wave 0 nears the task's end: a unit claimed early is held back from
            // workers that free up first
            const int32_t due = wave0_tiles + max(n0 - kClaimLead, 0);
            while (uni(__hip_atomic_load(&sh.started, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) < due)
                __builtin_amdgcn_s_sleep(2);
            int32_t c = 0;
            if (lane == 0) c = __hip_atomic_fetch_add(a.counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            live = open(a.workers + uni(c), false);
        } else {
            live = open(after, false);
        }
        wave0_tiles += n0;
    }
    // The last worker to finish puts the claim counter back to zero for the next launch
    // (relaxed: see for_each_task).  Only schedules that claim move it: without a task, 512
    // workers' atomics on one word would delay the others' first loads by ~3 us.
    if (dynamic && a.done_counter && lane == 0) {
        const int32_t done = __hip_atomic_fetch_add(a.done_counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (done == a.workers - 1) {
            __hip_atomic_store(a.counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.done_counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// ------------------------------------------------------------------ kernel
template <int DT, bool CSR, int D, bool kOut, bool kPow2, Rest kRest, bool kPasses>
__global__ __launch_bounds__(PGeo<D>::kThreads, PGeo<D>::kWavesPerSimd) void k_attention_pipe(sgd_decode_args a) {
    using GG = PGeo<D>;
    constexpr int kTile = GG::kTile, kWaves = GG::kWaves;
    extern __shared__ __align__(16) char dyn_smem[];
    PipeShared<D> &sh = *reinterpret_cast<PipeShared<D> *>(dyn_smem);
    const int lane0 = threadIdx.x & 63, wave = uni(threadIdx.x >> 6);
    const int32_t G = a.query_heads / a.kv_heads;
    char *const sq = dyn_smem + sizeof(PipeShared<D>);
    float *const so = reinterpret_cast<float *>(sq + 2 * G * GG::kQRow);
    const PageMap<kPow2> pm(a.page_size);
    if (wave == kWaves) {
        helper_wave<CSR, D, kPow2>(a, sh, sq, G, lane0, pm);
        return;
    }
    const float scale2 = a.scale * kLog2e;
    const int32_t heads = kPasses ? pass_heads<D>(G) : G;  // kPasses: G > heads per merge pass
    // kRestColumns: groups up to 4; kRestOwn: 8 and 16 heads at D = 256
    const bool one_set = kRest == kNoRest ? merge_sets<D>(G) == 1 : kRest == kRestOwn;
    const int32_t row_heads = kRest == kRestColumns ? 2 * heads : heads;  // merge_heads

    auto read_slot = [&](int32_t k) {
        const Slot s = sh.slot[k & 1];
        return Slot{uni(s.task), uni(s.request), uni(s.split), uni(s.start), uni(s.end), uni(s.group), uni(s.ind0), 0};
    };
    TileRegs<D> r;
    Source src{};
    // The wave's first tile of slot t (task k): its source, and its indices from LDS.
    auto first_tile = [&](const Slot &t, int32_t k, int lane) {
        src.kbase = static_cast<const char *>(a.k) + t.group * (a.k_stride[2] * 2);
        src.vbase = static_cast<const char *>(a.v) + t.group * (a.v_stride[2] * 2);
        src.rows = CSR ? a.pages + t.ind0 : a.pages + (int64_t)t.request * a.pt_stride[0];
        src.tok = t.start + wave * kTile;
        src.end = t.end;
        const int32_t *ix = sh.idx[k & 1] + wave * kTile;
        const int m = lane & 15, j = lane >> 4;
#pragma unroll
        for (int h = 0; h < GG::kHalves; ++h) r.idx[h] = ix[16 * h + 4 * j + (m & 3)];
    };
    auto merge_rows = [&](int par) { return so + (one_set ? 0 : par) * kWaves * row_heads * GG::kORow; };
    // The waves' states of task t's heads h0 .., merged in wave order.  A request's first split also writes
    // its normalized rows to `out` (kOut: sgd_decode_args.out set) -- final for a single-split
    // request, overwritten by the merge otherwise.
    auto merge = [&](const Slot &t, int par, int h0, int lane) {
        const float *rows = merge_rows(par);
#pragma clang loop unroll(disable)
        for (int x = 64 * wave + lane; x < heads * D; x += 64 * kWaves) {
            const int h = h0 + (uint32_t)x / D, d = (uint32_t)x % D;
            float mm = -INFINITY;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) mm = fmaxf(mm, sh.m[par][w][h]);
            float dd = 0.f, acc = 0.f, rest = 0.f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const float f = __builtin_amdgcn_exp2f(sh.m[par][w][h] - mm);
                const float *o = rows + (w * row_heads + h - h0) * GG::kORow + merge_pos<D>(d);
                dd += sh.d[par][w][h] * f;
                acc += *o * f;
                if constexpr (kRest == kRestColumns) rest += o[heads * GG::kORow] * f;
            }
            if constexpr (kRest == kRestColumns) acc += finite(rest);
            const int64_t row = (int64_t)t.request * a.query_heads + t.group * G + h;
            const int64_t slot = row * a.max_splits + t.split;
            a.partial[slot * D + d] = acc / dd;
            if (d == 0) a.lse[slot] = (mm + __log2f(dd)) * kLn2;
            if (kOut && t.split == 0) static_cast<uint16_t *>(a.out)[row * D + d] = (uint16_t)from_f32<DT>(acc / dd);
        }
    };

    lds_barrier();  // task 0 is published
    Slot cur{}, nxt{};
    int32_t n1 = 0;          // the wave's tiles of nxt
    bool requested = false;  // nxt's first tile is on its way
    int32_t started = 0;
    auto read_next = [&](int32_t k) {
        nxt = read_slot(k);
        n1 = nxt.task < 0 ? 0 : wave_tiles<D>(nxt.start, nxt.end, wave);
    };
    read_next(0);
    for (int32_t k = 0;; ++k) {
        int lane = lane0;  // laundered per task: per-lane offsets are rebuilt, not held live
        asm volatile("" : "+v"(lane));
        const int par = k & 1;
        if (n1 > 0 && !requested) {
            first_tile(nxt, k, lane);
            issue_k<CSR, D>(a, src, pm, lane, r);
            __builtin_amdgcn_sched_barrier(0);
            issue_v<CSR, D>(a, src, pm, lane, r);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (k > 0) merge(cur, par ^ 1, G - heads, lane);
        if (nxt.task < 0) break;
        cur = nxt;
        const int32_t n0 = n1;
        const char *q = sq + (par * G + (lane & 15 & (G - 1))) * GG::kQRow + (lane >> 4) * 16;
        State<D, kRest> st;
        st.m = -INFINITY;
        st.den = 0.f;
#pragma unroll
        for (int b = 0; b < GG::kBlocks; ++b) {
            st.o[b] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (kRest == kRestOwn) st.rest[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        bool known = false;  // nxt holds task k + 1
        requested = false;
        int32_t tok = cur.start + wave * kTile;
        for (int32_t left = n0; left > 0; --left, tok += kTile * kWaves) {
            asm volatile("" : "+s"(left));  // no peeled copy of the loop body
            if (wave == 0) {
                ++started;
                if (lane == 0)
                    __hip_atomic_store(&sh.started, started, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            // The tile to request meanwhile: this task's next one; after its last, the next
            // task's first if the helper has published it; else once more the task's last row
            // (its indices are loaded already, 512 B), so that the loads need no branch.
            src.tok += kTile * kWaves;
            if (left == 1) {
                // kPasses: not beside O in registers through the earlier passes
                known = !kPasses &&
                        uni(__hip_atomic_load(&sh.seq[par ^ 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) ==
                            k + 2;
                if (known) {
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                    read_next(k + 1);
                    requested = n1 > 0;
                    if (requested) first_tile(nxt, k + 1, lane);
                }
            }
            tile_step<DT, CSR, D, kPow2, kRest>(a, r, sh.kstage[wave], q, min(kTile, cur.end - tok), scale2, src, pm,
                                                lane, st);
        }

        // ---- the wave's state to LDS, then the merge
        st.den += __shfl_xor(st.den, 16, 64);
        st.den += __shfl_xor(st.den, 32, 64);
        if constexpr (kRest == kRestOwn) {
            // Straight-line code that a launch's first task fetches: the clamps stay out of it.
            float top = 0.f;
#pragma unroll
            for (int b = 0; b < GG::kBlocks; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) top = fmaxf(top, __builtin_fabsf(st.o[b][i]));
            if (__builtin_expect(__ballot(top == INFINITY) != 0, 0)) {
#pragma unroll
                for (int b = 0; b < GG::kBlocks; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) st.rest[b][i] = finite(st.rest[b][i]);
            }
#pragma unroll
            for (int b = 0; b < GG::kBlocks; ++b) st.o[b] = st.o[b] + st.rest[b];
        }
        const int n = lane & 15, j = lane >> 4;
        if (j == 0) {
            sh.m[par][wave][n] = st.m;
            sh.d[par][wave][n] = st.den;
        }
        for (int32_t h0 = 0;; h0 += heads) {
            if (one_set) lds_barrier();  // the rows' last merge has read them
            // the lane's row: its column's head, or that head's remainders
            const int row = kRest != kRestColumns ? n - h0 : n & 8 ? heads + (n & 7) : n;
            if (kRest != kRestColumns ? n >= h0 && n < h0 + heads : (n & 7) < heads) {
                float *dst = merge_rows(par) + (wave * row_heads + row) * GG::kORow;
#pragma unroll
                for (int b = 0; b < GG::kBlocks; ++b)
                    *reinterpret_cast<f32x4 *>(dst + 128 * (b / GG::kRowDims) + 4 * GG::kRowDims * j +
                                               4 * (b % GG::kRowDims)) = st.o[b];
            }
            if (!kPasses || h0 + heads == G) break;  // the last pass is merged with the next task's rows in flight
            lds_barrier();
            merge(cur, par, h0, lane);
        }
        lds_barrier();  // every wave's state, and task k + 1
        if (!known) read_next(k + 1);
    }
}

template <int DT, bool CSR, int D, bool kOut, bool kPow2, Rest kRest, bool kPasses>
int launch_pipe_o(const sgd_decode_args &a, hipStream_t stream) {
    static bool attr[kOnceDevices] = {};
    const int bytes = pipe_lds_bytes<D>(a.query_heads / a.kv_heads);
    if (int rc = set_dynamic_lds((const void *)k_attention_pipe<DT, CSR, D, kOut, kPow2, kRest, kPasses>, 80 * 1024, attr,
                                 "pipelined attention"))
        return rc;
    hipLaunchKernelGGL((k_attention_pipe<DT, CSR, D, kOut, kPow2, kRest, kPasses>), dim3(a.workers),
                       dim3(PGeo<D>::kThreads), bytes, stream, a);
    return launch_status("persistent_decode(pipelined)");
}

template <int DT, bool CSR, int D, bool kOut, bool kPow2>
int launch_pipe_g(const sgd_decode_args &a, hipStream_t stream) {
    const int g = a.query_heads / a.kv_heads;
    if (rest_form<D>(g) == kRestColumns)
        return launch_pipe_o<DT, CSR, D, kOut, kPow2, kRestColumns, false>(a, stream);
    if constexpr (D == 256)
        return g > pass_heads<D>(g) ? launch_pipe_o<DT, CSR, D, kOut, kPow2, kRestOwn, true>(a, stream)
                                    : launch_pipe_o<DT, CSR, D, kOut, kPow2, kRestOwn, false>(a, stream);
    else
        return launch_pipe_o<DT, CSR, D, kOut, kPow2, kNoRest, false>(a, stream);
}

// A power-of-two page (CSR's page of one token included) maps tokens by shift and mask;
// any other page size by division, in a separate build.
template <int DT, bool CSR, int D, bool kOut>
int launch_pipe_p(const sgd_decode_args &a, hipStream_t stream) {
    if constexpr (CSR) return launch_pipe_g<DT, CSR, D, kOut, true>(a, stream);
    else
        return (a.page_size & (a.page_size - 1)) == 0 ? launch_pipe_g<DT, CSR, D, kOut, true>(a, stream)
                                                      : launch_pipe_g<DT, CSR, D, kOut, false>(a, stream);
}

template <int DT, bool CSR, int D>
int launch_pipe_d(const sgd_decode_args &a, hipStream_t stream) {
    return a.out ? launch_pipe_p<DT, CSR, D, true>(a, stream) : launch_pipe_p<DT, CSR, D, false>(a, stream);
}

template <int DT, bool CSR>
int launch_pipe_t(const sgd_decode_args &a, hipStream_t stream) {
    switch (a.head_dim) {
        case 64: return launch_pipe_d<DT, CSR, 64>(a, stream);
        case 256: return launch_pipe_d<DT, CSR, 256>(a, stream);
        default: return launch_pipe_d<DT, CSR, 128>(a, stream);
    }
}

}  // namespace

int launch_attention_pipe(const sgd_decode_args &a, hipStream_t stream) {
    if (a.dtype == SGD_BF16)
        return a.csr ? launch_pipe_t<SGD_BF16, true>(a, stream) : launch_pipe_t<SGD_BF16, false>(a, stream);
    return a.csr ? launch_pipe_t<SGD_FP16, true>(a, stream) : launch_pipe_t<SGD_FP16, false>(a, stream);
}

}  // namespace sgd
