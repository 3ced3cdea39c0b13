// The decode step's writes around the attention, in one launch: the new tokens' K and
// V rows into the layer's KV pool at their cache slots (what the reference adapter's
// token_to_kv_pool.set_kv_buffer does, integrations/sglang_backend.py:91-92) and the
// step's q rows into the engine's stable per-layer query buffer (the qbuf.copy_ of
// :102-103).  Upstream these are three device operations per layer (two scatters and
// a copy); here one launch moves each token's 2 x Hkv x D + Hq x D 16-bit values
// as 16-byte vector copies.
//
// The data is copied bit for bit (no dtype conversion); K/V rows go to the pool with
// ordinary stores (the next step's attention reads them), q rows likewise.  A slot
// outside [0, cache_tokens) is skipped: a kernel cannot raise the way torch's
// index_put does, so the host checks what it can and the device never writes out of
// bounds.
#include "common.h"

namespace sgd {
namespace {

constexpr int kStoreThreads = 256;
// Workgroups of a launch, unless the batch alone is more: beyond them a token's workgroups loop over its
// pieces (768 tokens of 64 / 8 heads: 5.6 us, 6.1 with a workgroup for every 256 pieces, 6.0 with a
// limit of 1024; 512 tokens of 32 / 8 heads: 3.9, 4.1 with a limit of 2048).
constexpr int kStoreGroups = 1536;

struct StoreArgs {
    const char *k_new, *v_new;   // [batch, Hkv, D] (may be null: no KV write)
    char *k_cache, *v_cache;     // [cache_tokens, Hkv, D]
    const void *loc;             // [batch] slot per token, int32 or int64
    const char *q_in;            // [batch, Hq, D] (may be null: no q staging)
    char *q_out;                 // [>= batch, Hq, D]
    int64_t kn[2], vn[2], kc[2], vc[2], qi[2], qo[2];  // byte strides of dims 0 and 1
    int64_t cache_tokens;
    int32_t batch, hkv, hq, chunks;  // chunks: 16-byte pieces per (token, head) row
    int32_t loc64;
};

// Where one kind of rows (K, V or q) comes from and goes to for a token: its row in both, and the
// stride between heads.
struct Rows {
    const char *src;
    char *dst;
    int64_t from, to;
};

// Latency-bound while the pieces fit the chip (12 KB per token at the 8B shape): one 16-byte piece per
// thread, so that a token's pieces are one round trip, made together with its slot's.  With one
// workgroup per token looping over them it was a round trip for the slot and one per 256 pieces (one token,
// 32 / 8 heads: 2.7 us, now 2.3).  With thousands of tokens the address arithmetic counts: a wave
// whose pieces are of one kind has their strides in scalar registers (1024 tokens of 32 / 8 heads:
// 5.1 us; 5.6 with the strides loaded per lane and without the limit above; 4.9 with one workgroup
// per token).
__global__ __launch_bounds__(kStoreThreads) void k_store_kv_stage_q(StoreArgs a) {
    const int32_t b = blockIdx.x;
    const int32_t kv_pieces = a.k_new ? a.hkv * a.chunks : 0;
    const int32_t q_pieces = a.q_in ? a.hq * a.chunks : 0;
    int64_t slot = -1;
    if (kv_pieces) {
        slot = a.loc64 ? static_cast<const int64_t *>(a.loc)[b] : static_cast<const int32_t *>(a.loc)[b];
        if (slot >= a.cache_tokens) slot = -1;
    }
    const Rows k{a.k_new + b * a.kn[0], a.k_cache + slot * a.kc[0], a.kn[1], a.kc[1]};
    const Rows v{a.v_new + b * a.vn[0], a.v_cache + slot * a.vc[0], a.vn[1], a.vc[1]};
    const Rows q{a.q_in + b * a.qi[0], a.q_out + b * a.qo[0], a.qi[1], a.qo[1]};
    // pieces [0, kv) are K rows, [kv, 2 kv) V rows, then q rows; piece = (head, chunk)
    const int64_t pieces = 2 * (int64_t)kv_pieces + q_pieces;
    for (int64_t p = (int64_t)blockIdx.y * kStoreThreads + threadIdx.x; p < pieces;
         p += (int64_t)gridDim.y * kStoreThreads) {
        const int kind = p < kv_pieces ? 0 : p < 2 * (int64_t)kv_pieces ? 1 : 2;
        const int32_t r = (int32_t)(p - kind * (int64_t)kv_pieces);
        const int32_t h = (int32_t)((uint32_t)r / (uint32_t)a.chunks), c = r - h * a.chunks;
        auto copy = [&](const Rows &x) {
            const uint4 w = *reinterpret_cast<const uint4 *>(x.src + h * x.from + c * 16);
            if (kind == 2 || slot >= 0) *reinterpret_cast<uint4 *>(x.dst + h * x.to + c * 16) = w;
        };
        const int first = __builtin_amdgcn_readfirstlane(kind);
        if (__ballot(kind != first) != 0) {
            auto pick = [&](auto x, auto y, auto z) { return kind == 0 ? x : kind == 1 ? y : z; };
            copy(Rows{pick(k.src, v.src, q.src), pick(k.dst, v.dst, q.dst), pick(k.from, v.from, q.from),
                      pick(k.to, v.to, q.to)});
        } else if (first == 0) {
            copy(k);
        } else if (first == 1) {
            copy(v);
        } else {
            copy(q);
        }
    }
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace sgd

using namespace sgd;

extern "C" int sgd_store_kv_stage_q(const void *k_new, const void *v_new, const int64_t *new_strides,
                                    const void *loc, int32_t loc_is_int64, void *k_cache, void *v_cache,
                                    const int64_t *cache_strides, int64_t cache_tokens, const void *q_in,
                                    const int64_t *q_in_strides, void *q_out, const int64_t *q_out_strides,
                                    int32_t batch, int32_t kv_heads, int32_t query_heads, int32_t head_dim,
                                    int32_t dtype, void *stream) {
    if (dtype != SGD_BF16 && dtype != SGD_FP16) return einval("store_kv_stage_q: dtype %d", dtype);
    if (batch < 0 || kv_heads <= 0 || query_heads <= 0 || (head_dim * 2) % 16 != 0 || head_dim <= 0)
        return einval("store_kv_stage_q: batch %d, heads %d/%d, head_dim %d", batch, query_heads, kv_heads,
                      head_dim);
    const bool kv = k_new != nullptr, q = q_in != nullptr;
    if (kv && (!v_new || !new_strides || !loc || !k_cache || !v_cache || !cache_strides || cache_tokens <= 0))
        return einval("store_kv_stage_q: KV write needs k/v, their strides, loc and both caches");
    if (q && (!q_out || !q_in_strides || !q_out_strides))
        return einval("store_kv_stage_q: q staging needs q_in, q_out and their strides");
    StoreArgs a{};
    a.batch = batch;
    a.hkv = kv_heads;
    a.hq = query_heads;
    a.chunks = head_dim * 2 / 16;
    a.loc64 = loc_is_int64 != 0;
    a.cache_tokens = cache_tokens;
    // element strides (dims 0, 1; dim 2 has unit stride) -> byte strides, 16-byte aligned
    auto bytes = [](const int64_t *s, int64_t *out) {
        out[0] = s[0] * 2;
        out[1] = s[1] * 2;
        return (out[0] % 16) == 0 && (out[1] % 16) == 0 && s[0] >= 0 && s[1] >= 0;
    };
    if (kv) {
        a.k_new = static_cast<const char *>(k_new);
        a.v_new = static_cast<const char *>(v_new);
        a.k_cache = static_cast<char *>(k_cache);
        a.v_cache = static_cast<char *>(v_cache);
        a.loc = loc;
        if (!bytes(new_strides, a.kn) || !bytes(new_strides + 2, a.vn) || !bytes(cache_strides, a.kc) ||
            !bytes(cache_strides + 2, a.vc))
            return einval("store_kv_stage_q: K/V strides must be non-negative multiples of 8 elements");
        if (!aligned16(k_new) || !aligned16(v_new) || !aligned16(k_cache) || !aligned16(v_cache))
            return einval("store_kv_stage_q: K/V rows must be 16-byte aligned");
    }
    if (q) {
        a.q_in = static_cast<const char *>(q_in);
        a.q_out = static_cast<char *>(q_out);
        if (!bytes(q_in_strides, a.qi) || !bytes(q_out_strides, a.qo))
            return einval("store_kv_stage_q: q strides must be non-negative multiples of 8 elements");
        if (!aligned16(q_in) || !aligned16(q_out)) return einval("store_kv_stage_q: q rows must be 16-byte aligned");
    }
    if (batch == 0 || (!kv && !q)) return 0;
    clear_stale_error();
    const int64_t pieces = (int64_t)a.chunks * ((kv ? 2 * (int64_t)kv_heads : 0) + (q ? query_heads : 0));
    const int64_t parts = (pieces + kStoreThreads - 1) / kStoreThreads;
    const int64_t most = batch < kStoreGroups ? kStoreGroups / batch : 1;
    hipLaunchKernelGGL(k_store_kv_stage_q, dim3(batch, (unsigned)(parts < most ? parts : most)), dim3(kStoreThreads), 0,
                       (hipStream_t)stream, a);
    return launch_status("store_kv_stage_q");
}
