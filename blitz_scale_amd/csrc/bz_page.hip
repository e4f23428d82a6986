// KV page writes for gfx950: prefill store and decode append, each optionally fused with the
// Llama rotate-half RoPE of the new K rows and of the matching q rows, and with e4m3
// quantisation for an fp8 pool.  Replaces src/kernel/page.cu of the BlitzScale worker; pool
// helpers replace the allocation at src/blitz/cache_manager.h:136-142 and the layer pointer
// bump at src/model/llama.h:378-381.
#include <algorithm>
#include <cmath>

#include "bz_common.hpp"

namespace bz {

struct PageWriteArgs {
    char* k_data;
    char* v_data;
    const int32_t* indices;
    const int32_t* indptr;
    const int32_t* last_page_len;
    const int32_t* steps_ahead; // optional: the table is this many decode steps ahead of the present
    const void* k_src;
    const void* v_src;
    void* q_inout;
    const int32_t* ragged_indptr; // prefill only
    const float* k_scale;
    const float* v_scale;
    uint64_t stride_page, stride_n, stride_h;
    uint32_t batch_size, page_size, num_kv_heads, num_qo_heads, num_tokens;
    uint64_t tokens_per_wg;   // prefill only: four bits per 1024 tokens of the call, see page_write_kernel
    uint32_t rows_reciprocal, rows_held;
    int rope;
    RopeFreqs freqs;
};

// Prefill store, HBM-bound.  A workgroup takes up to kPwTokens consecutive tokens and moves all their rows (q heads to
// rotate in place, then the k heads, then the v heads).  A row of D elements is handled by D/16 lanes; each lane owns 8
// elements of the lower half and the 8 elements of the upper half that form rotate-half pairs with them.
//
// What bounds it with few rows per token is not the bytes but the chain in front of the stores: which request a token
// belongs to, its pages, the page id.  The rows do not depend on any of that, so they are asked for early and the chain
// runs while they travel: the entries of the ragged index (64 at a time, a lane compares one, the wave counts) go out in
// front of the rows, and the rest is scalar where the tokens are one request's.  Several tokens share one such chain.
// Against one token per workgroup, a binary search and then the rows (bf16, K rotated in place, buffers that are in no
// cache): 12 700 tokens of 8 heads 47.6 -> 26.8 us (4.7 TB/s), 28 000 93.5 -> 54.9, 28 231 of 40 heads (1.45 GB) 262 -> 259
// (5.6 TB/s), 8 192 requests of two tokens 52.6 -> 29.8, 8 000 empty requests in front of 192 58 -> 30, 300 tokens as
// before.  Where the call rotates 64 q heads in place beside 8 kv heads it is slower, 126 -> 130 us for 16 000 tokens.
//
// Rows a lane holds at a time: one (76 registers, six waves per SIMD), or three where a token has 64 rows or more, q is
// not among them and the pool is of the rows' type (12 700 tokens of 8 heads 26.8 us with one, 27.7 with three; 20 000 of 16 heads 74.5 / 79; 16 000 of 64 q and 8
// kv heads 130 / 131, in f16 131 / 137; 20 000 of 32 heads 155 / 152; 28 231 of 40 263 / 258; into an fp8 pool 9 000 of 32 53.9 / 58.9, of 40 67.4 / 72.0).
// Where a token fills a workgroup, sharing has nothing to give, and some calls are slower than with one token each and no
// rows asked for in front: one request into an fp8 pool (the two above 49.5 and 61), copies of 28 231 tokens of 32 heads 226
// -> 236 us and of 40 289 -> 297, k and q of 40 heads rotated in place 500 -> 513; the same fp8 calls with 16 requests are faster
// (28 231 of 32 heads 280 -> 239, of 40 347 -> 309).
constexpr int kPwRowsFew = 1, kPwRowsMany = 3;
constexpr int kPwTokens = 16;   // most tokens of a workgroup

// A first request so that the one that token n belongs to, the last b with ragged[b] <= n (ragged[0] = 0, n < ragged[batch]),
// is among the 64 from it on: every round the wave looks at 64 entries of what is left.
__device__ __forceinline__ int narrow_requests(const int32_t* __restrict__ ragged, int batch, int n) {
    const int lane = threadIdx.x & 63;
    int lo = 0, count = batch;
    while (count > 64) {
        const int stride = (count + 63) / 64, at = lane * stride;
        const unsigned long long le = __ballot(at < count && ragged[lo + min(at, count - 1)] <= n);
        const int k = max((int)__popcll(le), 1) - 1;
        lo += k * stride;
        count = min(stride, count - k * stride);
    }
    return lo;
}
// entry first + lane of the ragged index; past the last request none that a token could reach
__device__ __forceinline__ int request_entry(const int32_t* __restrict__ ragged, int batch, int first) {
    const int i = first + (threadIdx.x & 63), e = ragged[min(i, batch)];
    return i < batch ? e : INT32_MAX;
}
__device__ __forceinline__ int entries_up_to(int entry, int n) { return __builtin_popcountll(__ballot(entry <= n)); }

template <typename ST, typename PT, int D, int HELD> // HELD: rows a lane holds at a time
__global__ __launch_bounds__(256) void page_write_kernel(const int32_t* __restrict__ ragged, const int32_t* __restrict__ indptr,
                                                         const int32_t* __restrict__ indices, PageWriteArgs a) {
    constexpr int LANES = D / 16, ROWS = 256 / LANES; // ROWS: rows the workgroup handles side by side
    __shared__ float2 s_cs[kPwTokens][D / 2];
    const int lane = threadIdx.x % LANES, wave_lane = threadIdx.x & 63;
    const int B = (int)a.batch_size, Hkv = (int)a.num_kv_heads, P = (int)a.page_size;
    const int Hq = (a.rope && a.q_inout) ? (int)a.num_qo_heads : 0;
    const bool in_place = a.rope && (Hq > 0 || a.rope == 2); // the caller's k rows are rotated as well
    const int R = Hq + 2 * Hkv;
    // (the count that the call names is only an upper bound, and BZ_NUM_TOKENS_FROM_INDPTR is the largest one: how many
    // tokens a workgroup takes goes by the tokens that there are)
    const int rows_end = (int)min((uint32_t)max(ragged[B], 0), a.num_tokens);
    const int T = 1 + (int)((a.tokens_per_wg >> (4 * min(max(rows_end / 1024, 1) - 1, 15))) & 15);
    for (int n0 = (int)blockIdx.x * T; n0 < rows_end; n0 += (int)gridDim.x * T) {
        const int nt = min(T, rows_end - n0), rows = nt * R;
        // What decides the request goes out in front of the rows -- loads return in order -- and what hangs on it is
        // scalar where the tokens are one request's, which does not wait for the rows either.
        const int first = B > 64 ? narrow_requests(ragged, B, n0) : 0;
        const int entry = request_entry(ragged, B, first + 1);
        __builtin_amdgcn_sched_barrier(0);
        // row r of the workgroup: token r / R (by the reciprocal the host made: exact, r < 2^16), row r % R of it
        auto token_of = [&](int r) { return (int)__umulhi((uint32_t)r, a.rows_reciprocal); };
        auto src_of = [&](int r, int t) -> ST* {
            const int hr = r - t * R;
            const size_t tok = (size_t)(n0 + t);
            if (hr < Hq) return reinterpret_cast<ST*>(a.q_inout) + (tok * a.num_qo_heads + hr) * D;
            const bool is_k = hr < Hq + Hkv;
            const void* base = is_k ? a.k_src : a.v_src;
            return reinterpret_cast<ST*>(const_cast<void*>(base)) + (tok * Hkv + (is_k ? hr - Hq : hr - Hq - Hkv)) * D;
        };
        Vec8<ST> lo[HELD], hi[HELD];
        auto load_rows = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < HELD; ++i) {
                const int r = min(r0 + i * ROWS, rows - 1); // (past the end: the last row again, not stored)
                const ST* src = src_of(r, token_of(r));
                lo[i].load(src + lane * 8);
                hi[i].load(src + D / 2 + lane * 8);
            }
        };
        int r0 = (int)threadIdx.x / LANES;
        load_rows(r0);

        __builtin_amdgcn_sched_barrier(0);
        // ---- where the tokens go: lane t of every wave has token n0 + t.
        // A request longer than the pages its table row lists (the reference asserts seq_len >= append length,
        // src/kernel/page.cu:43): the tokens without a page are not cached -- nothing is written outside the listed
        // pages -- but a call that rotates q / k in place still rotates their rows, so that the attention call which
        // follows sees every row of the request rotated alike.
        int pos, slot, page = -1; // page < 0: the token is not cached
        const int after = entries_up_to(entry, n0), b = first + after;
        const int pos0 = n0 - ragged[b], pg0 = pos0 / P, slot0 = pos0 - pg0 * P;
        const bool one_request = __builtin_amdgcn_readlane(entry, min(after, 63)) >= n0 + nt;
        if (one_request && slot0 + nt <= 2 * P) { // of one or two pages
            const int ip = indptr[b], np = indptr[b + 1] - ip;
            const int page0 = pg0 < np ? indices[ip + pg0] : -1;
            const int page1 = slot0 + nt > P && pg0 + 1 < np ? indices[ip + pg0 + 1] : -1;
            pos = pos0 + wave_lane;
            slot = slot0 + wave_lane;
            page = slot < P ? page0 : page1;
            if (slot >= P) slot -= P;
        } else {
            int mine = b;
            const int next = request_entry(ragged, B, b + 1);
            const bool far = entries_up_to(next, n0 + nt - 1) == 64; // (a run of empty requests longer than that)
            for (int t = 1; t < nt; ++t) {
                int bt = b + entries_up_to(next, n0 + t);
                if (far) {
                    const int from = narrow_requests(ragged, B, n0 + t);
                    bt = from + entries_up_to(request_entry(ragged, B, from + 1), n0 + t);
                }
                if (wave_lane == t) mine = bt;
            }
            pos = n0 + wave_lane - ragged[mine];
            const int ip = indptr[mine], np = indptr[mine + 1] - ip, pg = pos / P;
            slot = pos - pg * P;
            if (wave_lane < nt && pg < np) page = indices[ip + pg];
        }
        const bool live = page >= 0 || in_place; // (without a page it is at least rotated)
        if (a.rope) {
            __syncthreads(); // the previous pass has finished with the table
            constexpr int TW = 256 / (D / 2); // tokens whose angles are worked out side by side
            for (int t = (int)threadIdx.x / (D / 2); t < nt; t += TW) {
                const int p = __shfl(pos, t, 64);
                float s, c;
                sincosf((float)p * a.freqs.f[threadIdx.x % (D / 2)], &s, &c);
                s_cs[t][threadIdx.x % (D / 2)] = make_float2(c, s);
            }
            __syncthreads();
        }
        for (;;) {
#pragma unroll
            for (int i = 0; i < HELD; ++i) {
                const int r = r0 + i * ROWS;
                const int t = token_of(min(r, rows - 1)), hr = r - t * R;
                const int64_t row_page = __shfl(page, t, 64);
                const int row_slot = __shfl(slot, t, 64);
                const bool row_live = __shfl((int)live, t, 64) != 0;
                if (r >= rows || !row_live) continue;
                const bool is_q = hr < Hq, is_k = !is_q && hr < Hq + Hkv;
                const int h = is_k ? hr - Hq : hr - Hq - Hkv;
                const bool rotate = (is_q || is_k) && a.rope;
                const float* scale = is_q ? nullptr : (is_k ? a.k_scale : a.v_scale);
                // Pages written at prefill are next read by a later decode step, long after they have left the
                // caches: non-temporal stores leave the cache to the caller's q / k / v rows, which the attention
                // call reads next (16 prompts of 128..4096 tokens, 40 heads: 362 -> 353 us).
                PT* dst = reinterpret_cast<PT*>(is_k ? a.k_data : a.v_data) +
                          ((size_t)row_page * a.stride_page + (size_t)row_slot * a.stride_n + (size_t)h * a.stride_h);
                if constexpr (sizeof(ST) == sizeof(PT)) {
                    if (!rotate && !scale) { // bit-exact copy
                        if (row_page < 0) continue;
                        Vec8<PT> l2, h2;
                        l2.raw = lo[i].raw;
                        h2.raw = hi[i].raw;
                        l2.store_nt(dst + lane * 8);
                        h2.store_nt(dst + D / 2 + lane * 8);
                        continue;
                    }
                }
                float x[8], y[8];
                lo[i].to_float(x);
                hi[i].to_float(y);
                if (rotate) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float2 cs = s_cs[t][lane * 8 + e];
                        float xr, yr;
                        rope_pair(x[e], y[e], cs.x, cs.y, xr, yr);
                        x[e] = xr;
                        y[e] = yr;
                    }
                }
                if (is_q || (is_k && in_place)) {
                    // rotated in place: q, and in the fused RoPE of the prefill path the caller's k rows as well, so
                    // that the attention call that follows contracts rotated q with rotated k
                    ST* src = src_of(r, t);
                    Vec8<ST> lr, hr2;
                    lr.from_float(x);
                    hr2.from_float(y);
                    lr.store(src + lane * 8);
                    hr2.store(src + D / 2 + lane * 8);
                }
                if (is_q || row_page < 0) continue;
                if (scale) {
                    const float sc = scale[h];
#pragma unroll
                    for (int e = 0; e < 8; ++e) { x[e] = x[e] / sc; y[e] = y[e] / sc; }
                }
                Vec8<PT> l2, h2;
                l2.from_float(x);
                h2.from_float(y);
                l2.store_nt(dst + lane * 8);
                h2.store_nt(dst + D / 2 + lane * 8);
            }
            r0 += HELD * ROWS;
            if (r0 - (int)threadIdx.x / LANES >= rows) break; // (workgroup-uniform)
            load_rows(r0);
        }
    }
}

// Decode append: one workgroup per sequence, one new row per (q | k | v) head.  At decode batch sizes the
// kernel is nothing but its chain of dependent memory round trips, so everything that does not depend
// on the page table (the counter, the table entries themselves, the caller's q / k / v rows) is
// requested up front; the page id is the one dependent fetch and overlaps with the angles.
template <typename ST, typename PT, int D>
__global__ __launch_bounds__(256) void append_kernel(PageWriteArgs a) {
    constexpr int LANES = D / 16;
    constexpr int ROWS = 256 / LANES;
    constexpr int MAXR = 4; // rows per lane group held in registers; more rows take the loop at the end
    __shared__ float s_cos[D / 2], s_sin[D / 2];

    const int b = blockIdx.x;
    const int ahead = a.steps_ahead ? *a.steps_ahead : 0;
    const int ip0 = a.indptr[b], ip1 = a.indptr[b + 1];
    const int lpl = a.last_page_len[b];
    const int lane = threadIdx.x % LANES, r0 = threadIdx.x / LANES;
    const int Hq = (a.rope && a.q_inout) ? (int)a.num_qo_heads : 0;
    const int Hkv = (int)a.num_kv_heads;
    const int total_rows = Hq + 2 * Hkv;
    auto row_src = [&](int r) -> const ST* { // rows 0..Hq-1: q heads, then the k heads, then the v heads
        if (r < Hq) return reinterpret_cast<const ST*>(a.q_inout) + ((size_t)b * a.num_qo_heads + r) * D;
        const bool is_k = r < Hq + Hkv;
        return reinterpret_cast<const ST*>(is_k ? a.k_src : a.v_src) + ((size_t)b * Hkv + (is_k ? r - Hq : r - Hq - Hkv)) * D;
    };
    Vec8<ST> lo[MAXR], hi[MAXR];
#pragma unroll
    for (int i = 0; i < MAXR; ++i) {
        const int r = r0 + i * ROWS;
        if (r < total_rows) {
            const ST* src = row_src(r);
            lo[i].load(src + lane * 8);
            hi[i].load(src + D / 2 + lane * 8);
        }
    }
    const int np = ip1 - ip0;
    if (np <= 0) return;
    const int pos = (np - 1) * (int)a.page_size + lpl - 1 - max(ahead, 0);
    if (pos < 0) return; // the sequence has no token yet at the present step
    const int64_t page = a.indices[ip0 + pos / (int)a.page_size];
    const int slot = pos % (int)a.page_size;
    if (a.rope) {
        for (int i = threadIdx.x; i < D / 2; i += 256) {
            float s, c;
            sincosf((float)pos * a.freqs.f[i], &s, &c);
            s_cos[i] = c;
            s_sin[i] = s;
        }
        __syncthreads();
    }
    auto finish_row = [&](int r, Vec8<ST>& l, Vec8<ST>& h) {
        const bool is_q = r < Hq, is_k = !is_q && r < Hq + Hkv;
        const bool rotate = (is_q || is_k) && a.rope;
        float x[8], y[8];
        if (is_q || rotate || (is_k ? a.k_scale : a.v_scale) || sizeof(ST) != sizeof(PT)) {
            l.to_float(x);
            h.to_float(y);
        }
        if (rotate) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float c = s_cos[lane * 8 + e], sn = s_sin[lane * 8 + e];
                float xr, yr;
                rope_pair(x[e], y[e], c, sn, xr, yr);
                x[e] = xr;
                y[e] = yr;
            }
        }
        if (is_q) { // rotated in place
            ST* row = const_cast<ST*>(row_src(r));
            l.from_float(x);
            h.from_float(y);
            l.store(row + lane * 8);
            h.store(row + D / 2 + lane * 8);
            return;
        }
        const int hd = is_k ? r - Hq : r - Hq - Hkv;
        PT* dst = reinterpret_cast<PT*>(is_k ? a.k_data : a.v_data) +
                  ((size_t)page * a.stride_page + (size_t)slot * a.stride_n + (size_t)hd * a.stride_h);
        const float* scale = is_k ? a.k_scale : a.v_scale;
        Vec8<PT> l2, h2;
        if constexpr (sizeof(ST) == sizeof(PT)) {
            if (!rotate && !scale) { // bit-exact copy
                l2.raw = l.raw;
                h2.raw = h.raw;
                l2.store(dst + lane * 8);
                h2.store(dst + D / 2 + lane * 8);
                return;
            }
        }
        if (scale) {
            const float sc = scale[hd];
#pragma unroll
            for (int e = 0; e < 8; ++e) { x[e] = x[e] / sc; y[e] = y[e] / sc; }
        }
        l2.from_float(x);
        h2.from_float(y);
        l2.store(dst + lane * 8);
        h2.store(dst + D / 2 + lane * 8);
    };
#pragma unroll
    for (int i = 0; i < MAXR; ++i) {
        const int r = r0 + i * ROWS;
        if (r < total_rows) finish_row(r, lo[i], hi[i]);
    }
    for (int r = r0 + MAXR * ROWS; r < total_rows; r += ROWS) {
        Vec8<ST> l, h;
        const ST* src = row_src(r);
        l.load(src + lane * 8);
        h.load(src + D / 2 + lane * 8);
        finish_row(r, l, h);
    }
}

template <typename ST, typename PT, bool PREFILL>
static int launch_page_write_d(const PageWriteArgs& a, int D, uint32_t grid, hipStream_t s) {
    if (grid == 0) return 0;
    if constexpr (PREFILL) {
        auto launch = [&](auto kernel) { launch_kernel(kernel, dim3(grid), dim3(256), 0, s, a.ragged_indptr, a.indptr, a.indices, a); };
        if (D == 128) a.rows_held == kPwRowsMany ? launch(page_write_kernel<ST, PT, 128, kPwRowsMany>) : launch(page_write_kernel<ST, PT, 128, kPwRowsFew>);
        else if (D == 64) a.rows_held == kPwRowsMany ? launch(page_write_kernel<ST, PT, 64, kPwRowsMany>) : launch(page_write_kernel<ST, PT, 64, kPwRowsFew>);
        else return BZ_ERR_UNSUPPORTED;
    } else {
        if (D == 128) launch_kernel((append_kernel<ST, PT, 128>), dim3(grid), dim3(256), 0, s, a);
        else if (D == 64) launch_kernel((append_kernel<ST, PT, 64>), dim3(grid), dim3(256), 0, s, a);
        else return BZ_ERR_UNSUPPORTED;
    }
    BZ_LAUNCH_CHECK();
    return 0;
}

template <bool PREFILL>
static int launch_page_write(const PageWriteArgs& a, int src_dtype, int pool_dtype, int D, uint32_t grid,
                             hipStream_t s) {
    if (src_dtype == BZ_F16 && pool_dtype == BZ_F16) return launch_page_write_d<f16_t, f16_t, PREFILL>(a, D, grid, s);
    if (src_dtype == BZ_BF16 && pool_dtype == BZ_BF16) return launch_page_write_d<bf16_t, bf16_t, PREFILL>(a, D, grid, s);
    if (src_dtype == BZ_F16 && pool_dtype == BZ_E4M3) return launch_page_write_d<f16_t, e4m3_t, PREFILL>(a, D, grid, s);
    if (src_dtype == BZ_BF16 && pool_dtype == BZ_E4M3) return launch_page_write_d<bf16_t, e4m3_t, PREFILL>(a, D, grid, s);
    return BZ_ERR_UNSUPPORTED;
}

static int fill_args(PageWriteArgs& a, const bz_paged_kv_t* kv, const void* k, const void* v, void* q_inout,
                     uint32_t num_qo_heads, int rope, float rope_theta, const float* k_scale, const float* v_scale,
                     bool prefill) {
    if (!kv || !k || !v || !kv->k_data || !kv->v_data) return BZ_ERR_BAD_ARG;
    if (!kv->indices || !kv->indptr || (!prefill && !kv->last_page_len)) return BZ_ERR_BAD_ARG;
    if (kv->stride_n % 8 || kv->stride_h % 8 || kv->stride_page % 8) return BZ_ERR_BAD_ARG;
    a.k_data = (char*)kv->k_data; a.v_data = (char*)kv->v_data;
    a.indices = kv->indices; a.indptr = kv->indptr; a.last_page_len = kv->last_page_len;
    a.steps_ahead = kv->steps_ahead;
    a.k_src = k; a.v_src = v; a.q_inout = q_inout; a.ragged_indptr = nullptr;
    a.k_scale = k_scale; a.v_scale = v_scale;
    a.stride_page = kv->stride_page; a.stride_n = kv->stride_n; a.stride_h = kv->stride_h;
    a.batch_size = kv->batch_size; a.page_size = kv->page_size; a.num_kv_heads = kv->num_kv_heads;
    a.num_qo_heads = num_qo_heads; a.num_tokens = 0;
    a.rope = rope == 2 ? 2 : (rope ? 1 : 0);
    a.freqs = make_rope_freqs((int)kv->head_dim, rope_theta > 0.f ? rope_theta : 1e4f);
    return 0;
}

// ---- one pass over the cached K rows of a page table: rotate them in place at their positions (direction +1) or
// take the rotation off again (direction -1).  A cache that arrives with K as the projection left it -- the
// reference's convention, whose decode call rotates every cached row at every step (attention_decode.cu:35) -- is
// brought to this library's convention (K cached rotated, the decode kernels rotate q only) once, at the speed of
// a copy, instead of paying for the rotation at every step; a cache that leaves for such a consumer is taken back.
// Workgroup (b, c) takes pages c, c + gridDim.y, ... of sequence b: the angles of a page's slots go through LDS
// (they are shared by the kv heads), eight lanes per row as in the page writes.
struct RopeCachedArgs {
    char* k_data;
    const int32_t* indices;
    const int32_t* indptr;
    const int32_t* last_page_len;
    uint64_t stride_page, stride_n, stride_h;
    uint32_t page_size, num_kv_heads;
    float direction;
    RopeFreqs freqs;
};

template <typename PT, int D>
__global__ __launch_bounds__(256) void rope_cached_k_kernel(RopeCachedArgs a) {
    extern __shared__ float2 s_cs[]; // [slot][pair]
    constexpr int LANES = D / 16;
    const int b = blockIdx.x;
    const int ip0 = a.indptr[b], np = a.indptr[b + 1] - ip0;
    if (np <= 0) return;
    const int P = (int)a.page_size, Hkv = (int)a.num_kv_heads;
    const int lane = threadIdx.x % LANES;
    for (int pg = blockIdx.y; pg < np; pg += gridDim.y) {
        const int slots = pg + 1 < np ? P : min(max(a.last_page_len[b], 0), P);
        const int64_t page = a.indices[ip0 + pg];
        __syncthreads(); // the previous page's angles are no longer read
        for (int i = threadIdx.x; i < slots * (D / 2); i += 256) {
            float sn, cs;
            sincosf((float)(pg * P + i / (D / 2)) * a.freqs.f[i % (D / 2)], &sn, &cs);
            s_cs[i] = make_float2(cs, a.direction * sn);
        }
        __syncthreads();
        for (int r = threadIdx.x / LANES; r < slots * Hkv; r += 256 / LANES) {
            const int slot = r / Hkv, h = r % Hkv;
            PT* row = reinterpret_cast<PT*>(a.k_data) +
                      ((size_t)page * a.stride_page + (size_t)slot * a.stride_n + (size_t)h * a.stride_h);
            Vec8<PT> lo, hi;
            lo.load(row + lane * 8);
            hi.load(row + D / 2 + lane * 8);
            float x[8], y[8];
            lo.to_float(x);
            hi.to_float(y);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float2 cs = s_cs[slot * (D / 2) + lane * 8 + e];
                float xr, yr;
                rope_pair(x[e], y[e], cs.x, cs.y, xr, yr);
                x[e] = xr;
                y[e] = yr;
            }
            lo.from_float(x);
            hi.from_float(y);
            lo.store(row + lane * 8);
            hi.store(row + D / 2 + lane * 8);
        }
    }
}

__global__ void steps_ahead_advance_kernel(int32_t* steps_ahead) {
    const int32_t v = *steps_ahead;
    if (v > 0) *steps_ahead = v - 1;
}

} // namespace bz

using namespace bz;

extern "C" int bz_steps_ahead_advance(int32_t* steps_ahead, void* stream) {
    if (!steps_ahead) return BZ_ERR_BAD_ARG;
    launch_kernel(steps_ahead_advance_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, steps_ahead);
    BZ_LAUNCH_CHECK();
    return 0;
}

extern "C" int bz_store_prefill_kv(const bz_paged_kv_t* kv, void* k, const void* v, int src_dtype,
                                   const int32_t* ragged_indptr, uint32_t num_tokens, void* q_inout,
                                   uint32_t num_qo_heads, int rope, float rope_theta, const float* k_scale,
                                   const float* v_scale, void* stream) {
    PageWriteArgs a;
    int rc = fill_args(a, kv, k, v, q_inout, num_qo_heads, rope, rope_theta, k_scale, v_scale, true);
    if (rc) return rc;
    if (!ragged_indptr) return BZ_ERR_BAD_ARG;
    a.ragged_indptr = ragged_indptr;
    a.num_tokens = num_tokens;
    if (kv->batch_size == 0) return 0;
    // Tokens per workgroup: the number whose rows fill the lanes best in one pass, but no more than leaves four workgroups
    // per compute unit: with fewer the chip idles, and a short call is over after one chain anyway.
    const uint32_t rows = (a.rope && q_inout ? num_qo_heads : 0) + 2 * kv->num_kv_heads; // of one token
    const bool counted = num_tokens != BZ_NUM_TOKENS_FROM_INDPTR;
    // (a launch of one workgroup per token would not exist for more: such a count is none)
    if (counted && num_tokens > UINT32_MAX / 256) return (int)hipErrorInvalidConfiguration;
    const bool supported = kv->head_dim == 128 || kv->head_dim == 64; // (others are refused below, where there is something to store)
    // (measured beside page_write_kernel)
    a.rows_held = (a.rope && q_inout) || rows < 64 || kv->kv_dtype != src_dtype ? kPwRowsFew : kPwRowsMany;
    uint32_t per_wg[kPwTokens]; // tokens of a workgroup when the call has 1024 (i + 1) of them
    for (uint32_t& t : per_wg) t = 1;
    if (supported && rows > 1) {
        const uint32_t held = a.rows_held * (256 / (kv->head_dim / 16));
        uint32_t T = 1;
        float best = 0.f;
        for (uint32_t t = 1; t <= kPwTokens; ++t) {
            const float filled = (float)(t * rows) / (float)((t * rows + held - 1) / held * held);
            if ((t == 1 || t * rows <= held) && filled > best + 0.01f) { best = filled; T = t; }
            per_wg[t - 1] = T;
        }
    }
    a.tokens_per_wg = 0;
    for (uint32_t i = 0; i < kPwTokens; ++i) a.tokens_per_wg |= (uint64_t)(per_wg[i] - 1) << (4 * i);
    a.rows_reciprocal = rows > 1 ? (uint32_t)(((1ull << 32) + rows - 1) / rows) : 0;
    // With the count known one workgroup per T tokens; otherwise (the reference's four-argument call,
    // src/kernel/page.h:66-67, whose launch is shaped by page size and batch alone, page.cu:84-89) a fixed launch whose
    // workgroups stride over the tokens that ragged_indptr[batch_size] counts.
    const uint32_t T = per_wg[std::min<uint32_t>(std::max(num_tokens / 1024, 1u) - 1, kPwTokens - 1)];
    const uint32_t grid = supported && rows == 0 ? 0 : (counted ? (num_tokens + T - 1) / T : 8192u);
    return launch_page_write<true>(a, src_dtype, kv->kv_dtype, (int)kv->head_dim, grid, (hipStream_t)stream);
}

extern "C" int bz_append_decode_kv(const bz_paged_kv_t* kv, const void* k, const void* v, int src_dtype,
                                   void* q_inout, uint32_t num_qo_heads, int rope, float rope_theta,
                                   const float* k_scale, const float* v_scale, void* stream) {
    PageWriteArgs a;
    int rc = fill_args(a, kv, k, v, q_inout, num_qo_heads, rope, rope_theta, k_scale, v_scale, false);
    if (rc) return rc;
    return launch_page_write<false>(a, src_dtype, kv->kv_dtype, (int)kv->head_dim, kv->batch_size,
                                    (hipStream_t)stream);
}

extern "C" int bz_rope_cached_k(const bz_paged_kv_t* kv, float rope_theta, int inverse, void* stream) {
    if (!kv || !kv->k_data || !kv->indices || !kv->indptr || !kv->last_page_len) return BZ_ERR_BAD_ARG;
    if (kv->stride_n % 8 || kv->stride_h % 8 || kv->stride_page % 8 || kv->page_size == 0) return BZ_ERR_BAD_ARG;
    if (kv->kv_dtype != BZ_F16 && kv->kv_dtype != BZ_BF16) return BZ_ERR_UNSUPPORTED; // (e4m3 rows would be requantised)
    const int D = (int)kv->head_dim;
    if (D != 128 && D != 64) return BZ_ERR_UNSUPPORTED;
    const size_t lds = (size_t)kv->page_size * (D / 2) * sizeof(float2);
    if (lds > 64 * 1024) return BZ_ERR_UNSUPPORTED; // page_size <= 128 (head_dim 128) / 256 (head_dim 64)
    if (kv->batch_size == 0) return 0;
    RopeCachedArgs a;
    a.k_data = (char*)kv->k_data;
    a.indices = kv->indices; a.indptr = kv->indptr; a.last_page_len = kv->last_page_len;
    a.stride_page = kv->stride_page; a.stride_n = kv->stride_n; a.stride_h = kv->stride_h;
    a.page_size = kv->page_size; a.num_kv_heads = kv->num_kv_heads;
    a.direction = inverse ? -1.0f : 1.0f;
    a.freqs = make_rope_freqs(D, rope_theta > 0.f ? rope_theta : 1e4f);
    const dim3 grid(kv->batch_size, 32);
    hipStream_t s = (hipStream_t)stream;
    if (kv->kv_dtype == BZ_F16) {
        if (D == 128) launch_kernel((rope_cached_k_kernel<f16_t, 128>), grid, dim3(256), lds, s, a);
        else launch_kernel((rope_cached_k_kernel<f16_t, 64>), grid, dim3(256), lds, s, a);
    } else {
        if (D == 128) launch_kernel((rope_cached_k_kernel<bf16_t, 128>), grid, dim3(256), lds, s, a);
        else launch_kernel((rope_cached_k_kernel<bf16_t, 64>), grid, dim3(256), lds, s, a);
    }
    BZ_LAUNCH_CHECK();
    return 0;
}

// ---- pool helpers -----------------------------------------------------------------------------
extern "C" void bz_paged_kv_set_layout(bz_paged_kv_t* kv, int layout) {
    const uint64_t H = kv->num_kv_heads, P = kv->page_size, D = kv->head_dim;
    kv->stride_page = 2 * H * P * D;
    if (layout == BZ_LAYOUT_HND) { kv->stride_n = D; kv->stride_h = P * D; }
    else { kv->stride_n = H * D; kv->stride_h = D; }
}

extern "C" uint64_t bz_kv_pool_bytes(uint32_t num_layers, uint64_t max_pages, uint32_t num_kv_heads,
                                     uint32_t page_size, uint32_t head_dim, int kv_dtype) {
    return (uint64_t)2 * num_layers * max_pages * num_kv_heads * page_size * head_dim * dtype_bytes(kv_dtype);
}

extern "C" int bz_kv_pool_alloc(void** base, uint64_t bytes) {
    if (!base) return BZ_ERR_BAD_ARG;
    return (int)hipMalloc(base, (size_t)bytes);
}

extern "C" int bz_kv_pool_free(void* base) { return (int)hipFree(base); }

extern "C" void bz_kv_layer_view(bz_paged_kv_t* kv, void* pool_base, uint32_t layer, uint64_t max_pages) {
    const uint64_t es = dtype_bytes(kv->kv_dtype);
    char* k = (char*)pool_base + (uint64_t)layer * max_pages * kv->stride_page * es;
    kv->k_data = k;
    kv->v_data = k + (kv->stride_page / 2) * es;
}

extern "C" const char* bz_build_info(void) { return "blitz-scale paged-attention path, gfx950, wave64"; }

extern "C" const char* bz_error_string(int code) {
    switch (code) {
        case 0: return "success";
        case BZ_ERR_BAD_ARG: return "bz: invalid argument";
        case BZ_ERR_UNSUPPORTED: return "bz: unsupported shape or type";
        case BZ_ERR_WORKSPACE: return "bz: workspace too small";
        case BZ_ERR_NOT_PLANNED: return "bz: plan() has not been called";
        case BZ_ERR_NO_PAGES: return "bz: out of KV pages";
        default: return hipGetErrorString((hipError_t)code);
    }
}
