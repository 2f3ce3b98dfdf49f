// The online count rows (tot, dist, cnt of every query under the step rule, exact_match/src/online.rs :259 counts) of a
// whole range of steps at once, with no step-by-step state (no counterpart in the reference's GPU libraries;
// ngram_amd/online.py drives it). A level's occurrences, listed in the order they begin to count in (ng_online_order's
// sort), have their rank in that order as their time: a step-s query counts exactly the occurrences of rank below
// lim(s) = those whose step is at most s. So with the occurrences of each context kept together in rank order,
//   tot  = its occurrences of rank < lim: a search of the context's ranks;
//   cnt  = the same among those followed by the query's own next token;
//   dist = its pairs whose first occurrence has rank < lim: a prefix sum over the context's occurrences that are the
//          first of their pair.
// Every occurrence is inserted once into the context table, its key slot << 16 | next sorted twice (by context and next
// token, and by context alone; stable, so ranks stay in order), and every query answered by searches: the work does not
// depend on the number of steps. Bound by the sorts (12 bytes read and written per occurrence and 8-bit pass) and the
// inserts' random lines; short streams by the launches. Measured, 262144 tokens in about 250 segments at n = 2..4: 14.0
// ms step by step (six launches a step), 1.27 ms here; 8.4M tokens in about 8200 segments: 468 ms and 9.4 ms.
#include "prim.h"
#include "probe.h"

namespace {

// Rank i's occurrence (ending at occ[i]; akey[i] its step, `none` past the last one): its context's slot (found or
// inserted) << 16 | next token, all ones of kbits bits where there is none, which sorts behind every pair.
template <int K>
__global__ void __launch_bounds__(256) oc_insert_k(const u16* __restrict__ tok, const u32* __restrict__ occ,
                                                   const u64* __restrict__ akey, u64 none, i64 n, int k, u64* ck,
                                                   u64 ccap, u64 kbits_ones, u64* __restrict__ key,
                                                   u32* __restrict__ val, u32* flags) {
    const i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x;
    if (i >= n) return;
    u64 out = kbits_ones;
    if (akey[i] != none) {
        const i64 g = occ[i];
        const i64 slot = ctx_find_insert(ck, ccap, qctx_key<K>(tok + g + 1, k), flags);
        if (slot >= 0) out = ((u64)slot << 16) | tok[g + 1];
    }
    key[i] = out;
    val[i] = (u32)i;
}

// first[rank] = 1 where that occurrence is its pair's first (ka / va: the occurrences sorted by pair).
__global__ void __launch_bounds__(256) oc_first_k(const u64* __restrict__ ka, const u32* __restrict__ va, i64 n,
                                                  u64 ones, unsigned char* __restrict__ first) {
    const i64 j = blockIdx.x * (i64)blockDim.x + threadIdx.x;
    if (j >= n) return;
    const u64 k = ka[j];
    first[va[j]] = k != ones && (j == 0 || ka[j - 1] != k) ? 1 : 0;
}

// Over the occurrences sorted by context (kb / vb): each context's bounds (start, end by slot), and f[j] = first of
// the occurrence at j (f[n] = 0: its exclusive sums then hold the total as well).
__global__ void __launch_bounds__(256) oc_bounds_k(const u64* __restrict__ kb, const u32* __restrict__ vb, i64 n,
                                                   u64 ones, const unsigned char* __restrict__ first,
                                                   u32* __restrict__ f, uint2* __restrict__ bounds) {
    const i64 j = blockIdx.x * (i64)blockDim.x + threadIdx.x;
    if (j > n) return;
    if (j == n || kb[j] == ones) {
        f[j] = 0;
        return;
    }
    const u64 slot = kb[j] >> 16;
    f[j] = first[vb[j]];
    if (j == 0 || kb[j - 1] >> 16 != slot) bounds[slot].x = (u32)j;
    if (j + 1 == n || kb[j + 1] >> 16 != slot) bounds[slot].y = (u32)(j + 1);
}

// Query i at position g = pos[i] (pos NULL: i), trained in step[g].
template <int K>
__global__ void __launch_bounds__(256) oc_query_k(const u16* __restrict__ tok, const int* __restrict__ avail,
                                                  const unsigned char* __restrict__ has_next,
                                                  const int* __restrict__ pos, i64 m, const u32* __restrict__ step,
                                                  const u64* __restrict__ akey, i64 n, int k,
                                                  const u64* __restrict__ ck, u64 ccap,
                                                  const uint2* __restrict__ bounds, const u32* __restrict__ vb,
                                                  const u32* __restrict__ pre, const u64* __restrict__ ka,
                                                  const u32* __restrict__ va, u32* __restrict__ tot,
                                                  u16* __restrict__ dist, u32* __restrict__ cnt, int nc, int ci) {
    const i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x;
    if (i >= m) return;
    const i64 g = pos ? pos[i] : i;
    if (avail[g] < ctx_len<K>(k)) return;
    const i64 slot = ctx_find(ck, ccap, qctx_key<K>(tok + g + 1, k));
    if (slot < 0) return;
    const u64 s = step[g];
    i64 lo = 0, hi = n;  // lim: the first rank whose step is past s (a wave's queries mostly share their step)
    while (lo < hi) {
        const i64 c = (lo + hi) >> 1;
        if (akey[c] <= s) lo = c + 1;
        else hi = c;
    }
    const u32 lim = (u32)lo;
    const uint2 ab = bounds[slot];
    u32 a = ab.x, b = ab.y;
    while (a < b) {
        const u32 c = (a + b) >> 1;
        if (vb[c] < lim) a = c + 1;
        else b = c;
    }
    if (a == ab.x) return;  // the context has not occurred yet
    const i64 at = g * nc + ci;
    const u32 d = pre[a] - pre[ab.x];
    u32 q = 0;
    if (has_next[g]) {
        const u64 want = ((u64)slot << 16) | tok[g + 1];
        u32 x = ab.x, e = ab.y;
        while (x < e) {
            const u32 c = (x + e) >> 1;
            if (ka[c] < want) x = c + 1;
            else e = c;
        }
        u32 y = x;
        e = ab.y;
        while (y < e) {
            const u32 c = (y + e) >> 1;
            if (ka[c] == want && va[c] < lim) y = c + 1;
            else e = c;
        }
        q = y - x;
    }
    tot[at] = a - ab.x;
    dist[at] = (u16)(d < 65535u ? d : 65535u);
    cnt[at] = q;
}

}  // namespace

// The occurrences of level k (occ[i] their last positions, akey[i] their steps ascending, `none` past the last of
// them: ng_online_order's output sorted) inserted into the context table ck (ccap slots, EMPTY-filled, below 2^cbits):
// key[i] = slot << 16 | next (2^(16 + cbits) - 1 where there is none), val[i] = i. flags[0] |= 2: the table is full.
extern "C" int ng_online_occ_insert(const u16* tok, const u32* occ, const u64* akey, u64 none, i64 n, int k, u64* ck,
                                    u64 ccap, int cbits, u64* key, u32* val, u32* flags, void* stream) {
    if (n < 1 || n > 0xFFFFFFFEll || !ccap || cbits < 1 || cbits > 40 || ccap >= (1ull << cbits) || !occ || !akey ||
        !ck || !key || !val || !flags)
        return -1;
    const u64 ones = (1ull << (16 + cbits)) - 1;
    LEVEL_DISPATCH(k, (oc_insert_k<K><<<grid_for(n, 256), 256, 0, (hipStream_t)stream>>>(tok, occ, akey, none, n, k, ck,
                                                                                        ccap, ones, key, val, flags)));
    return (int)hipGetLastError();
}

// From ng_online_occ_insert's pairs sorted stably by bits [0, 16 + cbits) (ka / va) and by bits [16, 16 + cbits) (kb /
// vb): bounds[slot] = the context's range in either (2 u32, only contexts that occur), pre[j] (n + 1 u32) = the pairs
// whose first occurrence lies before place j of the second. first: n bytes of scratch. CUB-style two-phase temp storage.
extern "C" int ng_online_occ_index(void* temp, size_t* temp_bytes, const u64* ka, const u32* va, const u64* kb,
                                   const u32* vb, i64 n, int cbits, unsigned char* first, u32* pre, u32* bounds,
                                   void* stream) {
    if (!temp_bytes || n < 1 || n > 0xFFFFFFFEll || cbits < 1 || cbits > 40) return -1;
    const size_t need = prim::scan_u32_temp_bytes(n + 1);
    if (!temp) {
        *temp_bytes = need;
        return 0;
    }
    if (*temp_bytes < need || !ka || !va || !kb || !vb || !first || !pre || !bounds) return -1;
    hipStream_t st = (hipStream_t)stream;
    const u64 ones = (1ull << (16 + cbits)) - 1;
    oc_first_k<<<grid_for(n, 256), 256, 0, st>>>(ka, va, n, ones, first);
    oc_bounds_k<<<grid_for(n + 1, 256), 256, 0, st>>>(kb, vb, n, ones, first, pre, (uint2*)bounds);
    int e = prim::exclusive_scan_u32(pre, pre, n + 1, nullptr, temp, st);
    return e ? e : (int)hipGetLastError();
}

// The queries at pos[0..m) (pos NULL: positions 0..m - 1), each of step[g], at level k: tot / dist / cnt of position
// g's row, column ci of [.., nc] arrays (left alone where the context is invalid or has not occurred by its step).
extern "C" int ng_online_occ_query(const u16* tok, const int* avail, const unsigned char* has_next, const int* pos,
                                   i64 m, const u32* step, const u64* akey, i64 n, int k, const u64* ck, u64 ccap,
                                   const u32* bounds, const u32* vb, const u32* pre, const u64* ka, const u32* va,
                                   u32* tot, u16* dist, u32* cnt, int nc, int ci, void* stream) {
    if (m < 0 || n < 1 || !ccap || nc < 1 || ci < 0 || ci >= nc || !avail || !has_next || !step || !akey || !ck ||
        !bounds || !vb || !pre || !ka || !va || !tot || !dist || !cnt)
        return -1;
    if (m == 0) return 0;
    LEVEL_DISPATCH(k, (oc_query_k<K><<<grid_for(m, 256), 256, 0, (hipStream_t)stream>>>(
                          tok, avail, has_next, pos, m, step, akey, n, k, ck, ccap, (const uint2*)bounds, vb, pre, ka, va,
                          tot, dist, cnt, nc, ci)));
    return (int)hipGetLastError();
}
