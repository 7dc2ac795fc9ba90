// ft_hip_grouped.hip -- one MoE layer for a batch of decode tokens with the
// (token, expert) pairs grouped by expert, so each routed expert's weights
// stream from HBM once for all of its tokens.
//
// The reference runs batched decode as one GEMV per pair over the pair list
// (ft-model/src/lib.rs:1507-1606: gemv_q4r_ptr per pair, gelu_mul_q8,
// gemv_q4r_ptr, reduce_pairs_weighted), re-reading an expert's weights for
// every token routed to it. Here:
//   router logits + top-k + q8(x)         (the launch-by-launch kernels)
//   k_group_pairs     one workgroup: pairs per expert, active-expert list (not in
//                     layers of up to 512 pairs on one family: their workgroups
//                     find their pairs in the routing)
//   k_grouped_gu      per (active expert, gate|up tile j): the tile's 64 rows
//                     in registers, dots against every token of the expert,
//                     GELU*up, q8 of the act block -> act[pair][j]
//   k_grouped_down    per (active expert, 128-row unit): y[pair][rows]
//   k_mfma_gu_tok, k_mfma_down_tok, k_mfma_down  the same two on the int8
//                     matrix cores, for batches of several tokens per expert
//   k_grouped_combine x_out[t] = x[t] + sum_k y[t*K+k] * w[t*K+k] in slot order
// Weights are in the fused layout (ft_hip_pack_experts_fused), so one packed
// bank serves this path and the batch-1 fused kernel.

#include "ft_device.hpp"
#include "ft_runtime.hpp"

#include <algorithm>
#include <type_traits>
#include <limits>

using namespace ft;

namespace {

constexpr int GT = 512;       // threads per workgroup
constexpr int GW = GT / 64;   // waves
constexpr int NT = 8;         // tokens per chunk of the gate|up kernel (LDS stays under 64 KB)
constexpr int NTD = 16;       // tokens per chunk of the down kernel
constexpr int DU = 16 * GW;   // rows per down unit (one 16-row tile per wave)
constexpr int MAX_PAIRS = 4096;
constexpr int MT = 16;        // tokens per MFMA tile

struct GroupWs {
    float* logits;      // [B][E]
    uint8_t* q8x;       // [B][H/32][40]
    int32_t* meta;      // [0] active experts; [1..] gexp[E], gstart[E], gcount[E]; [1+3E] MFMA groups
    int32_t* plist;     // [P] pairs grouped by expert
    int32_t* ppos;      // [P] token tiles of the MFMA groups (tile_entry)
    uint8_t* q8a;       // [P][I/32][40]
    uint8_t* q8m;       // the MFMA groups' act quants by group position q: [I/32][4][P] (qs words g, g+4), then [I/32][P] (d, qsum)
    float* ydn;         // [P][H]
    float* inv;         // [B] input RMS norm scales
    size_t bytes;
};

GroupWs group_ws(void* base, int64_t B, int64_t H, int64_t I, int64_t E, int64_t K) {
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    const int64_t P = B * K;
    size_t off = 0;
    GroupWs w{};
    uint8_t* p = (uint8_t*)base;
    w.logits = (float*)(p + off); off += up(sizeof(float) * B * E);
    w.q8x = p + off; off += up((size_t)B * (H / 32) * Q8_BLK);
    w.meta = (int32_t*)(p + off); off += up(sizeof(int32_t) * (2 + 3 * E));
    w.plist = (int32_t*)(p + off); off += up(sizeof(int32_t) * P);
    w.ppos = (int32_t*)(p + off); off += up(sizeof(int32_t) * P);
    w.q8a = p + off; off += up((size_t)P * (I / 32) * Q8_BLK);
    w.q8m = p + off; off += up((size_t)P * (I / 32) * Q8_BLK);
    w.ydn = (float*)(p + off); off += up(sizeof(float) * P * H);
    w.inv = (float*)(p + off); off += up(sizeof(float) * B);
    w.bytes = off;
    return w;
}

// Global -> LDS copy of n 32-bit items: item i is ld(i), stored by st(i, v).
// Each thread issues up to R loads before its first store, so the copy
// costs ceil(n / (R * GT)) load latencies rather than ceil(n / GT).
template <int R, typename Ld, typename St>
__device__ __forceinline__ void stage(int n, Ld ld, St st) {
    const int t = threadIdx.x;
    for (int base = 0; base < n; base += R * GT) {
        uint32_t v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = base + r * GT + t;
            v[r] = i < n ? ld(i) : 0u;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = base + r * GT + t;
            if (i < n) st(i, v[r]);
        }
    }
}

// Pairs p = t*K + k grouped by expert ids[p]. The order inside a group does
// not matter: every (row, token) dot is independent and outputs are written
// to the pair's own slot, so results are the same for any order.
// Groups are numbered with the experts of >= n_mfma tokens first (meta[1 +
// 3E] of them, for the MFMA kernels), then the others (for the dot4
// kernels), each in expert order. The MFMA groups' token tiles (up to
// MT tokens of one group each) are listed in ppos[0..P) as tile_entry
// words.
//
// TOPK (E <= 32 as launched): the routing itself first, from the logits (the
// arithmetic of k_topk_router, so the same ids and weights): 1024/E tokens
// per round, one thread per logit ranking it by rank_key among its token's
// E, then the softmax over each token's K in rank order; ids/wts written to
// ids_out/wts_out and kept in LDS for the grouping.
// A token tile: the number of tiles (up to 4096: 13 bits, in every entry), its
// group (10 bits) and its first token / MT (8 bits).
__host__ __device__ __forceinline__ uint32_t tile_entry(int n_tiles, int g, int c0) {
    return (uint32_t)n_tiles << 18 | (uint32_t)g << 8 | (uint32_t)c0 / MT;
}

template <bool TOPK>
__global__ __launch_bounds__(1024) void k_group_pairs(const int32_t* ids, int P, int E, int n_mfma, int32_t* meta,
                                                      int32_t* plist, int32_t* ppos, const float* logits,
                                                      const float* escale, int32_t* ids_out, float* wts_out, int K) {
    __shared__ int cnt[1024];
    __shared__ int scan[1024];
    __shared__ int act[1024];
    __shared__ int big[1024];
    __shared__ int sid[TOPK ? MAX_PAIRS : 1];
    __shared__ uint64_t key[TOPK ? 1024 : 1];
    __shared__ float sv[TOPK ? 1024 : 1], selv[TOPK ? 1024 : 1], exv[TOPK ? 1024 : 1];
    __shared__ int seli[TOPK ? 1024 : 1];
    const int t = threadIdx.x;
    if constexpr (TOPK) {
        const int B = P / K, TPR = 1024 / E;  // tokens per round
        const int slot = t / E, e = t - slot * E;
        const int ss = t / K, rr = t - ss * K;  // softmax: token slot ss, rank rr
        for (int r0 = 0; r0 < B; r0 += TPR) {
            const bool on = slot < TPR && r0 + slot < B;
            if (on) {
                const float v = logits[(int64_t)(r0 + slot) * E + e];
                sv[t] = v;
                key[t] = rank_key(v, e);
            }
            __syncthreads();
            if (on) {
                const uint64_t kt = key[t];
                const uint64_t* kr = key + slot * E;
                int rank = 0;
                for (int i0 = 0; i0 < E; i0 += 16) {  // 16 keys per step, their LDS reads issued together
                    uint64_t c[16];
#pragma unroll
                    for (int q = 0; q < 16; ++q) c[q] = kr[min(i0 + q, E - 1)];
#pragma unroll
                    for (int q = 0; q < 16; ++q) rank += (i0 + q < E && c[q] > kt) ? 1 : 0;
                }
                if (rank < K) {
                    selv[slot * K + rank] = sv[t];
                    seli[slot * K + rank] = e;
                }
            }
            __syncthreads();
            const bool on2 = ss < TPR && r0 + ss < B;
            if (on2) exv[t] = expf_libm(selv[t] - selv[ss * K]);
            __syncthreads();
            if (on2) {
                float denom = 0.0f;
                for (int j = 0; j < K; ++j) denom = denom + exv[ss * K + j];
                float w = exv[t] / denom;
                const int id = seli[t];
                if (escale) w = w * escale[id];
                const int p = (r0 + ss) * K + rr;
                ids_out[p] = id;
                wts_out[p] = w;
                sid[p] = id;
            }
            __syncthreads();
        }
    }
    auto pid = [&](int p) { return TOPK ? sid[p] : ids[p]; };
    for (int e = t; e < E; e += 1024) cnt[e] = 0;
    __syncthreads();
    // a thread's pairs, their experts and places in registers (P <= MAX_PAIRS)
    int ex[MAX_PAIRS / 1024], at[MAX_PAIRS / 1024];
#pragma unroll
    for (int i = 0; i < MAX_PAIRS / 1024; ++i) {
        if (i * 1024 >= P) break;
        const int p = i * 1024 + t;
        ex[i] = p < P ? min(max(pid(p), 0), E - 1) : 0;
    }
#pragma unroll
    for (int i = 0; i < MAX_PAIRS / 1024; ++i) {
        if (i * 1024 >= P) break;  // uniform
        if (i * 1024 + t < P) at[i] = atomicAdd(&cnt[ex[i]], 1);
    }
    __syncthreads();
    // inclusive prefix sums of counts and of "active" / "big" flags (E <=
    // 1024): within each wavefront by shuffles, then each thread adds the
    // totals of the wavefronts before its own (integer sums: exact in any order)
    const int c = t < E ? cnt[t] : 0;
    const bool vbig = c > 0 && c >= n_mfma;
    const int my_tiles = vbig ? (c + MT - 1) / MT : 0;
    // two sums to a word: pairs (up to 4096, 13 bits) and active experts, MFMA groups (up to 1024, 11 bits) and tiles
    int s0 = c | (c > 0) << 13, s1 = (int)vbig | my_tiles << 11;
    const int lane = t & 63, wv = t >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int n0 = __shfl_up(s0, d), n1 = __shfl_up(s1, d);
        if (lane >= d) {
            s0 += n0;
            s1 += n1;
        }
    }
    __shared__ int wtot[2][16];
    __shared__ int n_tiles;
    if (lane == 63) {
        wtot[0][wv] = s0;
        wtot[1][wv] = s1;
    }
    __syncthreads();
    for (int q = 0; q < wv; ++q) {
        s0 += wtot[0][q];
        s1 += wtot[1][q];
    }
    const int vc = s0 & 0x1FFF, va = s0 >> 13, vf = s1 & 0x7FF, vt = s1 >> 11;
    if (t == 1023) n_tiles = vt;
    scan[t] = vc;
    act[t] = va;
    big[t] = vf;
    __syncthreads();
    if (t < E && c > 0) {
        const int g = c >= n_mfma ? big[t] - 1 : big[1023] + (act[t] - big[t]) - 1;
        meta[1 + g] = t;                 // gexp
        meta[1 + E + g] = scan[t] - c;   // gstart
        meta[1 + 2 * E + g] = c;         // gcount
    }
    if (t == 0) {
        meta[0] = act[1023];
        meta[1 + 3 * E] = big[1023];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MAX_PAIRS / 1024 && i * 1024 < P; ++i)
        if (i * 1024 + t < P) plist[scan[ex[i]] - cnt[ex[i]] + at[i]] = i * 1024 + t;
    // the tile list (every tile holds a pair, so P entries suffice)
    for (int k = 0; k < my_tiles; ++k) ppos[vt - my_tiles + k] = (int32_t)tile_entry(n_tiles, big[t] - 1, k * MT);
    if (t == 0 && n_tiles == 0) ppos[0] = 0;
}

// The pairs p < P routed to expert e (ids[p] == e), ascending, into lst
// (LDS, at most SCAN_MAX); returns their count (the same in every thread).
// Lets a layer whose experts all take the dot4 kernels skip the grouping
// launch: each (tile, expert) workgroup finds its expert's pairs itself.
constexpr int SCAN_MAX = 1024;
__device__ __forceinline__ int scan_pairs(const int32_t* ids, int P, int e, int* lst, int* wcnt) {
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    int total = 0;
    for (int base = 0; base < P; base += GT) {
        const int p = base + t;
        const bool m = p < P && ids[p] == e;
        const uint64_t bal = __ballot(m);
        if (lane == 0) wcnt[wv] = __popcll(bal);
        __syncthreads();
        int off = total, sum = 0;
#pragma unroll
        for (int q = 0; q < GW; ++q) {
            off += q < wv ? wcnt[q] : 0;
            sum += wcnt[q];
        }
        if (m) lst[off + __popcll(bal & ((1ull << lane) - 1))] = p;
        total += sum;
        __syncthreads();  // wcnt is rewritten in the next round
    }
    return total;
}

// Gate|up tile j of active expert g for all of its tokens, then GELU*up and
// the q8 of act block j per token. BPW = H/32/8 blocks per wave. in_scale
// (input RMS norm, or null): a token's gate|up sums are first multiplied by
// in_scale[token]. SCAN: the grid's y is the expert, or a pair if there are
// fewer of those (5 tokens of the Gemma shape: 110 of 880 workgroups find
// nothing to do, of one row per expert 2,046 of 2,816), and the workgroup finds
// its expert's pairs in ids[0..P) (scan_pairs) instead of the group list.
template <int BPW, bool REC, bool SCAN>
__global__ __launch_bounds__(GT, 2) void k_grouped_gu(const uint8_t* bank, int64_t expert_bytes, const int32_t* meta,
                                                      const int32_t* plist, const uint8_t* q8x, uint8_t* q8a,
                                                      float* dbg_gu, const float* in_scale, int H, int I, int E,
                                                      int K, int n_mfma, int32_t* rec, const int32_t* ids, int P) {
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ int slst[SCAN ? SCAN_MAX : 1];
    __shared__ int wcnt[GW];
    const int nb = H >> 5, nbj = I >> 5;
    const int j = blockIdx.x;
    int e, n;
    const int32_t* lst;
    if constexpr (SCAN) {
        // fewer pairs than experts: the grid's y is a pair, and the expert's first pair takes the expert
        const bool by_pair = P < E;
        e = by_pair ? min(max(ids[blockIdx.y], 0), E - 1) : (int)blockIdx.y;
        n = scan_pairs(ids, P, e, slst, wcnt);
        if (n == 0 || (by_pair && slst[0] != (int)blockIdx.y)) return;
        lst = slst;
    } else {
        const int g = blockIdx.y + meta[1 + 3 * E];  // after the MFMA kernels' groups
        if (g >= meta[0]) return;
        e = meta[1 + g];
        n = meta[1 + 2 * E + g];
        if (n >= n_mfma) return;
        lst = plist + meta[1 + E + g];
    }
    // LDS: x q8 of NT tokens as [NT][nb][8 words] qs + [NT][nb] (d, qsum) pairs;
    // wave partial sums [GW][NT][64]; row sums [NT][64]; act [NT][32]
    uint4* xq = reinterpret_cast<uint4*>(lds);
    int2* xp = reinterpret_cast<int2*>(lds + NT * nb * 32);
    float* red = reinterpret_cast<float*>(lds + NT * nb * 40);
    float* rows = red + GW * NT * 64;
    float* actv = rows + NT * 64;
    uint32_t* ablk = reinterpret_cast<uint32_t*>(actv + NT * 32);
    const int t = threadIdx.x, wave = t >> 6, r = t & 63, b0 = wave * BPW;
    uint4 qv[BPW];
    uint32_t sc[BPW];
    {
        const uint8_t* T = bank + (int64_t)e * expert_bytes + (int64_t)j * nb * 1152;
#pragma unroll
        for (int i = 0; i < BPW; ++i) qv[i] = *reinterpret_cast<const uint4*>(T + nb * 128 + (b0 + i) * 1024 + r * 16);
#pragma unroll
        for (int i = 0; i < BPW; ++i) sc[i] = *reinterpret_cast<const uint16_t*>(T + (b0 + i) * 128 + r * 2);
    }
    __shared__ int ctok[NT];
    __shared__ float cscl[NT];  // the tokens' input-norm scales, loaded with the chunk's staging
    for (int c0 = 0; c0 < n; c0 += NT) {
        const int nt = min(NT, n - c0);
        __syncthreads();  // the previous chunk's LDS is consumed
        if (t < nt) ctok[t] = lst[c0 + t] / K;
        __syncthreads();
        {  // x q8 of this chunk's tokens: every load issued before the first store
            constexpr int W = 80 * BPW;  // q8 words per token (nb = 8 * BPW blocks of 10)
            constexpr int MW = (W + GT - 1) / GT;
            // an opaque thread index: the LDS offsets below are not hoisted
            // out of the chunk loop (they would stay live through the dots)
            int tq = t;
            asm volatile("" : "+v"(tq));
            uint32_t v[NT][MW];
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) {
                const uint32_t* src =
                    reinterpret_cast<const uint32_t*>(q8x + (int64_t)ctok[min(tt, nt - 1)] * nb * Q8_BLK);
#pragma unroll
                for (int m = 0; m < MW; ++m) {
                    const int wi = tq + m * GT;
                    v[tt][m] = (tt < nt && wi < W) ? src[wi] : 0u;
                }
            }
            const float sct = in_scale && t < nt ? in_scale[ctok[t]] : 1.0f;  // with the row loads
            if (t < NT) cscl[t] = sct;
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
                for (int m = 0; m < MW; ++m) {
                    const int wi = tq + m * GT, b = wi / 10, wd = wi - b * 10;
                    if (tt < nt && wi < W) {
                        if (wd >= 2) reinterpret_cast<uint32_t*>(xq)[(tt * nb + b) * 8 + (wd - 2)] = v[tt][m];
                        else reinterpret_cast<uint32_t*>(xp)[(tt * nb + b) * 2 + wd] = v[tt][m];
                    }
                }
            }
        }
        __syncthreads();
#pragma unroll 1
        for (int tt = 0; tt < nt; ++tt) {
            // one token at a time (not unrolled), its blocks' LDS reads in
            // batches of four blocks. The weights pass through an opaque move per token:
            // their nibble masks and f32 scales are not hoisted out of the
            // token loop, where they would take ~100 more registers.
            float acc = 0.0f;
#pragma unroll
            for (int i = 0; i < BPW; ++i)
                asm volatile("" : "+v"(qv[i].x), "+v"(qv[i].y), "+v"(qv[i].z), "+v"(qv[i].w), "+v"(sc[i]));
#pragma unroll
            for (int i = 0; i < BPW; ++i) {
                if (i % 4 == 0 && i > 0) __builtin_amdgcn_sched_barrier(0);
                const int xb = tt * nb + b0 + i;
                const int2 dq = xp[xb];
                const int dot = block_dot_v(qv[i], xq[xb * 2], xq[xb * 2 + 1], dq.y);
                acc = fmaf((float)dot, h2f((uint16_t)sc[i]) * __int_as_float(dq.x), acc);
                if constexpr (REC) {  // test record: the block's int32 dot
                    const int row = r < 32 ? j * 32 + r : I + j * 32 + (r - 32);
                    rec[((int64_t)lst[c0 + tt] * 2 * I + row) * nb + b0 + i] = dot;
                }
            }
            red[(wave * NT + tt) * 64 + r] = acc;
        }
        __syncthreads();
        for (int i = t; i < nt * 64; i += GT) {  // (token, row) sums over the waves, in wave order
            const int tt = i >> 6, rr = i & 63;
            float sv = 0.0f;
#pragma unroll
            for (int v = 0; v < GW; ++v) sv = sv + red[(v * NT + tt) * 64 + rr];
            if (in_scale) sv = sv * cscl[tt];
            rows[tt * 64 + rr] = sv;
            if (dbg_gu) {
                const int p = lst[c0 + tt];
                const int row = rr < 32 ? j * 32 + rr : I + j * 32 + (rr - 32);
                dbg_gu[(int64_t)p * 2 * I + row] = sv;
            }
        }
        __syncthreads();
        for (int i = t; i < nt * 32; i += GT) {
            const int tt = i >> 5, cc = i & 31;
            actv[tt * 32 + cc] = gelu_tanh(rows[tt * 64 + cc]) * rows[tt * 64 + 32 + cc];
        }
        __syncthreads();
        if (t < 4 * nt) quantize_block_quad(actv + (t >> 2) * 32, t & 3, ablk + (t >> 2) * 10);
        __syncthreads();
        for (int i = t; i < nt * 10; i += GT) {
            const int tt = i / 10, wd = i - tt * 10;
            const int p = lst[c0 + tt];
            reinterpret_cast<uint32_t*>(q8a + ((int64_t)p * nbj + j) * Q8_BLK)[wd] = ablk[tt * 10 + wd];
        }
    }
}

// Down rows 128u..128u+127 of active expert g (one 16-row tile per wave;
// thread (rr, s4) holds row rr's blocks s4, s4+4, ...) for all of its tokens.
// SCAN: as k_grouped_gu's.
template <int DB, bool REC, bool SCAN>
__global__ __launch_bounds__(GT, 1) void k_grouped_down(const uint8_t* bank, int64_t expert_bytes, int64_t gu_bytes,
                                                        const int32_t* meta, const int32_t* plist, const uint8_t* q8a,
                                                        float* ydn, int H, int I, int E, int n_mfma, int32_t* rec,
                                                        const int32_t* ids, int P) {
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ int slst[SCAN ? SCAN_MAX : 1];
    __shared__ int wcnt[GW];
    const int nbj = I >> 5;
    const int u = blockIdx.x;
    int e, n;
    const int32_t* lst;
    if constexpr (SCAN) {
        // fewer pairs than experts: the grid's y is a pair, and the expert's first pair takes the expert
        const bool by_pair = P < E;
        e = by_pair ? min(max(ids[blockIdx.y], 0), E - 1) : (int)blockIdx.y;
        n = scan_pairs(ids, P, e, slst, wcnt);
        if (n == 0 || (by_pair && slst[0] != (int)blockIdx.y)) return;
        lst = slst;
    } else {
        const int g = blockIdx.y + meta[1 + 3 * E];  // after the MFMA kernels' groups
        if (g >= meta[0]) return;
        e = meta[1 + g];
        n = meta[1 + 2 * E + g];
        if (n >= n_mfma) return;
        lst = plist + meta[1 + E + g];
    }
    uint4* aq = reinterpret_cast<uint4*>(lds);                  // [NTD][nbj][2 uint4]
    int2* ap = reinterpret_cast<int2*>(lds + NTD * nbj * 32);   // [NTD][nbj]
    const int t = threadIdx.x, wave = t >> 6, s4 = t & 3, rr = (t >> 2) & 15;
    const int dn_tile = nbj * 288;
    uint4 dq[DB];
    uint32_t dsc[DB];
    {
        const uint8_t* D = bank + (int64_t)e * expert_bytes + gu_bytes + (int64_t)(u * GW + wave) * dn_tile;
#pragma unroll
        for (int k = 0; k < DB; ++k) {
            const int b = min(s4 + 4 * k, nbj - 1);
            dq[k] = *reinterpret_cast<const uint4*>(D + nbj * 32 + b * 256 + rr * 16);
        }
#pragma unroll
        for (int k = 0; k < DB; ++k) {
            const int b = min(s4 + 4 * k, nbj - 1);
            dsc[k] = *reinterpret_cast<const uint16_t*>(D + b * 32 + rr * 2);
        }
    }
    for (int c0 = 0; c0 < n; c0 += NTD) {
        const int nt = min(NTD, n - c0);
        __syncthreads();
        stage<8>(  // act q8 of this chunk's pairs
            nt * nbj * 10,
            [&](int i) {
                const int tt = i / (nbj * 10), rem = i - tt * nbj * 10;
                const int p = lst[c0 + tt];
                return reinterpret_cast<const uint32_t*>(q8a + (int64_t)p * nbj * Q8_BLK)[rem];
            },
            [&](int i, uint32_t v) {
                const int tt = i / (nbj * 10), rem = i - tt * nbj * 10, b = rem / 10, wd = rem - b * 10;
                if (wd >= 2) reinterpret_cast<uint32_t*>(aq)[(tt * nbj + b) * 8 + (wd - 2)] = v;
                else reinterpret_cast<uint32_t*>(ap)[(tt * nbj + b) * 2 + wd] = v;
            });
        __syncthreads();
        for (int tt = 0; tt < nt; ++tt) {
            float acc = 0.0f;
#pragma unroll
            for (int k = 0; k < DB; ++k) {
                const int b = s4 + 4 * k;
                const int xb = tt * nbj + min(b, nbj - 1);
                const int2 pq = ap[xb];
                const int dot = block_dot_v(dq[k], aq[xb * 2], aq[xb * 2 + 1], pq.y);
                const float v = (float)dot * (h2f((uint16_t)dsc[k]) * __int_as_float(pq.x));
                acc = b < nbj ? acc + v : acc;
                if constexpr (REC) {  // test record: the block's int32 dot
                    if (b < nbj)
                        rec[((int64_t)lst[c0 + tt] * H + u * DU + wave * 16 + rr) * nbj + b] = dot;
                }
            }
            acc += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(acc), 0xB1, 0xF, 0xF, false));
            acc += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(acc), 0x4E, 0xF, 0xF, false));
            if (s4 == 0) {
                const int p = lst[c0 + tt];
                ydn[(int64_t)p * H + u * DU + wave * 16 + rr] = acc;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// int8 MFMA tile path, for groups of at least n_min tokens.
//
// v_mfma_i32_16x16x32_i8: D[16 rows][16 tokens] += A[16 rows][32] *
// B[32][16 tokens]; lane l holds A row l%16 and B column l%16 at k =
// 8*(l/16)..+7, and D rows 4*(l/16)..+3 of column l%16. One MFMA is one q4_0
// block (32 weights) of 16 rows against the q8 blocks of 16 tokens. The 32 k
// of a block are ordered so that lane group g = l/16 takes elements
// 4g..4g+3 and 16+4g..16+4g+3: for the weights the low and the high nibbles
// of qs word g (one dword, two masks), for the activations q8 words g and
// 4+g. The nibbles enter unsigned (0..15) and the accumulator starts at
// -8 * qsum of the token's block, so D is exactly the block's int32 dot
// sum (q-8)*q8 (ft-core/src/q4_0.rs:105-118). Per (row, token) the blocks
// then accumulate as acc = fma(float(D), d4 * d8, acc), in block order.
// ---------------------------------------------------------------------------
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

struct ActOp {
    long b;    // B operand: q8 words g and 4+g
    float d;   // the block's d
    int qsum;  // the block's sum of q
};

// Raw buffer loads: a per-lane 32-bit offset plus a uniform one (scalar
// register or immediate), so per-block addresses cost no vector registers;
// an offset past num_records reads 0.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

// A token's q8 block as the B operand of lane group g, from the q8m layout
// (GroupWs::q8m): q8 words (g, g+4) at vq + sq, {d, qsum} at vd + sd, one
// 8-byte load each. A lane without a token passes offsets past the buffer's
// end (NO_TOKEN; the buffer is smaller) and gets zeros.
constexpr uint32_t NO_TOKEN = 0x80000000u;
__device__ __forceinline__ ActOp act_op_m(__amdgpu_buffer_rsrc_t r, uint32_t vq, uint32_t vd, uint32_t sq,
                                          uint32_t sd) {
    const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(r, vq, sq, 0);
    const u32x2 dq = __builtin_amdgcn_raw_buffer_load_b64(r, vd, sd, 0);
    ActOp a;
    a.b = (long)(((uint64_t)w.y << 32) | w.x);
    a.d = __uint_as_float(dq.x);
    a.qsum = (int)dq.y;
    return a;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// A operand from qs word g of a row's block: low nibbles, then high nibbles.
__device__ __forceinline__ long nib_op(uint32_t w) {
    return (long)(((uint64_t)((w >> 4) & 0x0F0F0F0Fu) << 32) | (w & 0x0F0F0F0Fu));
}

// -8 * qsum of each token's block in the lanes and rows of a 16x16 tile, the
// accumulators' start for nib_op's unsigned nibbles: the block against rows of
// -8, one more instruction on the matrix cores (which the token-tile kernels leave idle
// most of the time) where a broadcast takes four on the VALU and qsum in LDS.
// (Signed operands 16 * (q - 8) and d8 / 16 need no start, but then a scale
// product below 2^-122 is rounded as a subnormal.)
__device__ __forceinline__ v4i start_sums(long bop) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8((long)0xF8F8F8F8F8F8F8F8ull, bop, v4i{0, 0, 0, 0}, 0, 0, 0);
}

// d4 * d8 of a 16x16 tile's (row, token) pairs, each rounded once as by
// v_mul_f32 (subnormals kept), in the lanes and order of the int8 MFMA's
// results: v_mfma_f32_4x4x1 is 16 outer products of 4 rows and 4 columns, one
// per lane quad. Lane (lg, li) gives the scale of row 4*lg + li%4 and its
// token's d. One instruction on the matrix cores (8 cycles) for four VALU ones.
__device__ __forceinline__ v4f scale_products(float d4, float d8) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(d4, d8, v4f{0, 0, 0, 0}, 0, 0, 0);
}

__device__ __forceinline__ v4i c_init(int qsum) {
    const int c = -8 * qsum;
    const v4i v = {c, c, c, c};
    return v;
}

// Four f16 scales (8 bytes) at p, widened.
__device__ __forceinline__ void scales4(const uint16_t* p, float (&sc)[4]) {
    const uint2 s2 = *reinterpret_cast<const uint2*>(p);
    sc[0] = h2f((uint16_t)(s2.x & 0xFFFF));
    sc[1] = h2f((uint16_t)(s2.x >> 16));
    sc[2] = h2f((uint16_t)(s2.y & 0xFFFF));
    sc[3] = h2f((uint16_t)(s2.y >> 16));
}

// A token tile found without the grouping launch (SCAN, up to TILE_SCAN pairs
// and 256 experts): the experts' tiles in expert order, a tile's pairs
// ascending. Every wave does it by itself, in LDS of its own (its LDS
// operations complete in order), so there is no barrier. For the down launch the
// workgroup of each tile's first act blocks leaves a record: expert | tokens << 16, then the
// 16 slots' pairs of 16 bits.
constexpr int TILE_SCAN = 512;
constexpr int TREC = 10;  // words per record (of GroupWs::q8a, a pair's act block, which a SCAN layer does not write)
struct TileScan {
    static constexpr int R = TILE_SCAN / 64;
    int ex[R];       // the experts of pairs r * 64 + lane
    int cn[4];       // the pair counts of experts 4 * lane ..
    int first, end;  // the tiles of these experts
    int e, c0, n;

    __device__ __forceinline__ static void order() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    }
    // Counts the pairs per expert (cnt: 256 words of the wave); the number of tiles.
    __device__ __forceinline__ int count(const int32_t* ids, int P, int E, int* cnt) {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int r = 0; r < R; ++r) ex[r] = r * 64 + lane < P ? min(max(ids[r * 64 + lane], 0), E - 1) : -1;
        *reinterpret_cast<int4*>(cnt + 4 * lane) = make_int4(0, 0, 0, 0);
        order();
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (ex[r] >= 0) atomicAdd(&cnt[ex[r]], 1);
        order();
        const int4 c = *reinterpret_cast<const int4*>(cnt + 4 * lane);
        cn[0] = c.x;
        cn[1] = c.y;
        cn[2] = c.z;
        cn[3] = c.w;
        int tiles = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) tiles += (cn[k] + MT - 1) / MT;
        end = tiles;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int u = __shfl_up(end, d);
            if (lane >= d) end += u;
        }
        first = end - tiles;
        return __builtin_amdgcn_readlane(end, 63);
    }
    // Tile k's expert, first token and the expert's token count, and its pairs into tok[MT].
    __device__ __forceinline__ void find(int k, int P, int* tok) {
        const int lane = threadIdx.x & 63;
        int at = first, ei = 0, ci = 0, ni = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int m = (cn[q] + MT - 1) / MT;
            const bool hit = k >= at && k < at + m;
            ei = hit ? 4 * lane + q : ei;
            ci = hit ? (k - at) * MT : ci;
            ni = hit ? cn[q] : ni;
            at += m;
        }
        const int src = __ffsll((unsigned long long)__ballot(k >= first && k < end)) - 1;
        e = __builtin_amdgcn_readlane(ei, src);
        c0 = __builtin_amdgcn_readlane(ci, src);
        n = __builtin_amdgcn_readlane(ni, src);
        int base = -c0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r * 64 >= P) break;  // uniform
            const uint64_t bal = __ballot(ex[r] == e);
            const int i = base + __popcll(bal & ((1ull << lane) - 1));
            if (ex[r] == e && i >= 0 && i < MT) tok[i] = r * 64 + lane;
            base += __popcll(bal);
        }
        order();
    }
};

// Gate|up of the MFMA groups by token tiles (up to 16 tokens of one expert): a
// workgroup takes one tile (of k_group_pairs' list, or with SCAN found by its
// waves) and NW consecutive act blocks j, one wave each (the 64 rows of gate|up
// tile j); the grid is one-dimensional over these units.
// The tokens' q8 rows are staged in LDS once, by block, so that a lane's
// operand words are one 8-byte read; a wave streams its tile's rows through a
// register ring of one K slice (BPW blocks, 1 KB per load), its scales
// through an LDS buffer of its own, and keeps all of a (row, token)'s sums:
// per slice acc = fma(float(D_b), d4_b * d8_b, acc) in block order, then the 8
// slice sums in order, the same bits as k_grouped_gu's. A lane holds
// gate and up of the same columns, so GELU*up and the act block's q8 stay in
// registers (two lane exchanges for the block's amax and sum), and go out as
// the q8m words they are.
//
// Why this form: the former kernel split K over the 8 waves of a workgroup,
// summed their partials through LDS for every 16 tokens and restaged the
// tokens' rows, an integer division and two dependent loads per word, at each
// tile of a group of over 16 tokens, on ranges of tiles that skewed token
// counts left uneven: 475 us for 512 tokens of the Gemma shape and 855 us for
// 173 zipf-skewed ones. Here a wave needs no other wave: 118-126 and 67 us.
// What bounds it: for many tokens the VALU (512 tokens: 63 instructions per
// block and wave, 71 % of the SIMDs' cycles, the matrix cores 24 %: 16
// conversions and 16 fmas are left after the scale products moved to the
// matrix cores, the others prepare operands or are the GELU epilogue); for few
// the weights (64 tokens: 285 MB in 63 us, 4.5 TB/s; the VALU 52 %). Blocks are consumed one at a
// time (sched_barrier), else the registers of a whole slice's dots spill.
// KS, for launches of few units: a workgroup is one act block, its 8 waves a
// slice each, and the first adds their sums in slice order, the same bits. The
// chain of a wave is an eighth as long: 16 tokens over 8 experts of H 4096, I 1024
// 104 -> 41 us a layer (against the 16-wave form), of H 2816, I 704 45 -> 34.
template <int BPW, int NW, int WPE, int D, int KH, bool REC, bool SCAN, bool KS>
__global__ __launch_bounds__(NW * 64, WPE) void k_mfma_gu_tok(
    const uint8_t* __restrict__ bank, int64_t expert_bytes, const int32_t* __restrict__ meta, uint32_t* tiles,
    const int32_t* __restrict__ plist, const uint8_t* __restrict__ q8x, uint8_t* q8m, float* dbg_gu,
    const float* __restrict__ in_scale, int I, int E, int K, int P, int32_t* rec, const int32_t* __restrict__ ids,
    uint32_t* trec) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int NB = 8 * BPW, TM = MT, NTH = NW * 64;
    constexpr int XS = TM * 8 + 2;  // words per block of the qs: a pad of two, so that lanes on consecutive blocks write distinct banks
    constexpr int NH = NB / KH, SH = 8 / KH;  // blocks and slices per staging of the tokens' rows
    constexpr int R = (TM * NH + NTH - 1) / NTH;  // (token, block) items staged per thread
    constexpr int SW = BPW * 128;   // bytes of a slice's scales
    static_assert(!KS || (NW == 8 && KH == 1), "a wave per slice");
    const int nbj = I >> 5, JG = KS ? nbj : (nbj + NW - 1) / NW;
    // workgroup id % 8 is the XCD: each takes a contiguous eighth of the (tile, act block group) units, so
    // the tiles of one expert, which read the same weights, run together behind one L2
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, li = t & 15, lg = lane >> 4;
    __shared__ __align__(16) int scnt[SCAN ? NW : 1][256], stok[SCAN ? NW : 1][MT];
    TileScan sc;
    const int n_tiles = SCAN ? sc.count(ids, P, E, scnt[wave]) : (int)(tiles[0] >> 18);
    const int n_units = n_tiles * JG, per = (n_units + 7) >> 3, ur = (int)blockIdx.x >> 3;
    const int unit = ((int)blockIdx.x & 7) * per + ur;
    if (ur >= per || unit >= n_units) return;
    const int jg = unit % JG;
    int e, c0, s0 = 0, nt;
    if constexpr (SCAN) {
        sc.find(unit / JG, P, stok[wave]);
        e = sc.e;
        c0 = sc.c0;
        nt = min(TM, sc.n - c0);
    } else {
        const uint32_t v0 = tiles[unit / JG];
        const int g = (int)(v0 >> 8) & 1023;
        c0 = (int)(v0 & 255) * MT;
        e = meta[1 + g];
        s0 = meta[1 + E + g];
        nt = min(TM, meta[1 + 2 * E + g] - c0);
    }
    auto pair = [&](int tt) __attribute__((always_inline)) { return SCAN ? stok[wave][tt] : plist[s0 + c0 + tt]; };
    const int jw = KS ? jg : jg * NW + wave, j = min(jw, nbj - 1), sl0 = KS ? wave : 0;  // sl0: the wave's first slice
    // LDS: the tokens' q8 words [NH][4 lane groups][TM] (g, g+4) | [NH][TM] d | the waves' slice scales
    uint32_t* xq = reinterpret_cast<uint32_t*>(lds);
    float* xd = reinterpret_cast<float*>(lds + (size_t)NH * XS * 4);
    uint8_t* scl = lds + (size_t)NH * (XS * 4 + TM * 4) + wave * SW;
    // the tokens' rows: thread item i = (token, block), 40 bytes
    uint2 st[R][5];
    auto load_act = [&](int h) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = r * NTH + t, tt = i / NH, b = i - tt * NH;
            if (tt < nt) {
                const uint2* src =
                    reinterpret_cast<const uint2*>(q8x + ((int64_t)(pair(tt) / K) * NB + h * NH + b) * Q8_BLK);
#pragma unroll
                for (int k = 0; k < 5; ++k) st[r][k] = src[k];
            }
        }
    };
    auto store_act = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = r * NTH + t, tt = i / NH, b = i - tt * NH;
            if (tt < nt) {
                uint32_t* q = xq + b * XS + tt * 2;
                *reinterpret_cast<uint2*>(q) = make_uint2(st[r][1].x, st[r][3].x);
                *reinterpret_cast<uint2*>(q + TM * 2) = make_uint2(st[r][1].y, st[r][3].y);
                *reinterpret_cast<uint2*>(q + TM * 4) = make_uint2(st[r][2].x, st[r][4].x);
                *reinterpret_cast<uint2*>(q + TM * 6) = make_uint2(st[r][2].y, st[r][4].y);
                xd[b * TM + tt] = __uint_as_float(st[r][0].x);
            }
        }
    };
    load_act(0);
    if (SCAN && jg == 0) {  // this tile's record, and the number of tiles
        if (t < MT / 2) {
            const uint32_t a = stok[0][min(2 * t, nt - 1)], b = stok[0][min(2 * t + 1, nt - 1)];
            trec[unit / JG * TREC + 1 + t] = a | b << 16;
        }
        if (t == 0) trec[unit / JG * TREC] = (uint32_t)e | (uint32_t)nt << 16;
        if (t == 0 && unit == 0) tiles[0] = tile_entry(n_tiles, 0, 0);
    }
    const uint8_t* T = bank + (int64_t)e * expert_bytes + (int64_t)j * NB * 1152;
    const __amdgpu_buffer_rsrc_t rs = buf_rsrc(T, NB * 128), rw = buf_rsrc(T + NB * 128, NB * 1024);
    const uint32_t vw16 = lg * 256 + li * 16;
    u32x4 aw[BPW], ss[2];
    auto load_scales = [&](int s) __attribute__((always_inline)) {  // the slice's scales, 16 bytes a lane and round
        ss[0] = __builtin_amdgcn_raw_buffer_load_b128(rs, lane * 16, s * SW, 0);
        ss[1] = __builtin_amdgcn_raw_buffer_load_b128(rs, min(1024 + lane * 16, SW - 16), s * SW, 0);
    };
    load_scales(sl0);
#pragma unroll
    for (int b = 0; b < D; ++b) aw[b] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw16, (sl0 * BPW + b) * 1024, 0);
    store_act();
    __syncthreads();
    if (KH == 1 && jw >= nbj) return;
    const int slot = min(li, nt - 1);  // this lane's token (past the end: the last one, never written)
    float tot[4][4];                   // [row tile][row]
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) tot[m][v] = 0.0f;
    auto slice = [&](int s, auto lastt) __attribute__((always_inline)) {
        constexpr bool last = decltype(lastt)::value;
        // the slice's scales into this wave's buffer (its reads of the slice before have all returned)
        asm volatile("" ::: "memory");
        *reinterpret_cast<u32x4*>(scl + lane * 16) = ss[0];
        if (1024 + lane * 16 < SW) *reinterpret_cast<u32x4*>(scl + 1024 + lane * 16) = ss[1];
        asm volatile("" ::: "memory");
        if (!last) load_scales(s + 1);
        float acc[4][4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[m][v] = 0.0f;
#pragma unroll
        for (int b = 0; b < BPW; ++b) {
            const int blk = s % SH * BPW + b;
            const uint2 q = *reinterpret_cast<const uint2*>(xq + blk * XS + (lg * TM + slot) * 2);
            const float ad = xd[blk * TM + slot];
            float dw[4];
#pragma unroll
            for (int m = 0; m < 4; ++m)
                dw[m] = h2f(*reinterpret_cast<const uint16_t*>(scl + b * 128 + m * 32 + lg * 8 + (li & 3) * 2));
            uint32_t w[4] = {aw[b].x, aw[b].y, aw[b].z, aw[b].w};
            quad_transpose(w[0], w[1], w[2], w[3]);
            if (b + D < BPW || !last)  // the block D ahead
                aw[(b + D) % BPW] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw16, (s * BPW + b + D) * 1024, 0);
            const long bop = (long)(((uint64_t)q.y << 32) | q.x);
            const v4i c8 = start_sums(bop);
            v4i d[4];
            v4f sp[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) sp[m] = scale_products(dw[m], ad);
#pragma unroll
            for (int m = 0; m < 4; ++m)
                d[m] = __builtin_amdgcn_mfma_i32_16x16x32_i8(nib_op(w[m]), bop, c8, 0, 0, 0);
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                if constexpr (REC) {  // test record: the (row, token) blocks' int32 dots
                    if (li < nt && jw < nbj)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const int rr = 16 * m + 4 * lg + v;
                            const int row = rr < 32 ? j * 32 + rr : I + j * 32 + (rr - 32);
                            rec[((int64_t)pair(slot) * 2 * I + row) * NB + s * BPW + b] = d[m][v];
                        }
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[m][v] = fmaf((float)d[m][v], sp[m][v], acc[m][v]);
                // the sums are formed here: left to the scheduler, the dots of a whole slice wait for theirs
                asm volatile("" : "+v"(acc[m][0]), "+v"(acc[m][1]), "+v"(acc[m][2]), "+v"(acc[m][3]));
            }
            __builtin_amdgcn_sched_barrier(0);  // one block's MFMA results live at a time
        }
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) tot[m][v] = tot[m][v] + acc[m][v];
    };
    if constexpr (KS) {
        slice(wave, std::true_type{});
        // the other waves' slice sums through LDS (over the tokens' rows), added in slice order by the first
        float4* part = reinterpret_cast<float4*>(lds);
        auto at = [&](int s, int m) { return (s * 64 + lane) * 4 + ((m + (lane >> 1)) & 3); };
        __syncthreads();
        if (wave > 0) {
#pragma unroll
            for (int m = 0; m < 4; ++m) part[at(wave, m)] = make_float4(tot[m][0], tot[m][1], tot[m][2], tot[m][3]);
        }
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int s = 1; s < 8; ++s)
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const float4 v = part[at(s, m)];
                tot[m][0] = tot[m][0] + v.x;
                tot[m][1] = tot[m][1] + v.y;
                tot[m][2] = tot[m][2] + v.z;
                tot[m][3] = tot[m][3] + v.w;
            }
    } else {
#pragma unroll 1
        for (int s = 0; s < 7; ++s) {
            if (KH > 1 && s == SH) {  // the rest of the tokens' rows, once every wave is done with the first part
                load_act(1);
                __syncthreads();
                store_act();
                __syncthreads();
            }
            slice(s, std::false_type{});
        }
        slice(7, std::true_type{});
    }
    if (KH > 1 && jw >= nbj) return;
    const int p = pair(slot), q = SCAN ? p : s0 + c0 + slot;
    const bool ok = li < nt;
    const float isc = in_scale ? in_scale[p / K] : 1.0f;
    float a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {  // columns 16*(i/4) + 4*lg + i%4 of the act block
        float gv = tot[i >> 2][i & 3], uv = tot[2 + (i >> 2)][i & 3];
        if (in_scale) {
            gv = gv * isc;
            uv = uv * isc;
        }
        if (dbg_gu && ok) {
            const int64_t o = (int64_t)p * 2 * I + j * 32 + (i >> 2) * 16 + lg * 4 + (i & 3);
            dbg_gu[o] = gv;
            dbg_gu[o + I] = uv;
        }
        a[i] = gelu_tanh(gv) * uv;
        __builtin_amdgcn_sched_barrier(0);  // one GELU's registers at a time
    }
    // the block's q8 over its four lanes (li + 16*lg), the arithmetic of quantize_block_quad
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(a[i]));
    amax = fmaxf(amax, __shfl_xor(amax, 16));
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    const float d = amax > 0.0f ? amax / 127.0f : 0.0f;
    const float inv = d > 0.0f ? 1.0f / d : 0.0f;
    int qsum = 0;
    uint32_t w[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int qi = (int)q8_clamp(roundf(a[i] * inv));
        qsum += qi;
        w[i >> 2] |= (uint32_t)(uint8_t)(int8_t)qi << (8 * (i & 3));
    }
    qsum += __shfl_xor(qsum, 16);
    qsum += __shfl_xor(qsum, 32);
    if (ok) {
        uint2* o = reinterpret_cast<uint2*>(q8m);
        o[(uint32_t)((j * 4 + lg) * P + q)] = make_uint2(w[0], w[1]);
        if (lg == 0) o[(uint32_t)(P * nbj * 4 + j * P + q)] = make_uint2(__float_as_uint(d), (uint32_t)qsum);
    }
}

// Down rows by token tiles, for rows of up to 4*NKB blocks: a wave takes 64
// rows (four 16-row tiles) of one expert for the up to 16 tokens of one token
// tile, workgroup unit (tile, NW waves of rows). The tokens' act words come
// from q8m as they lie (each block's words of a lane group contiguous over the
// group's tokens) and are staged in LDS once for the workgroup's waves; the
// rows stream through registers four blocks (NBUF - 1 batches) ahead. Per
// (row, token) acc = fma(float(D_b), d4_b * d8_b, acc) in block order, or with
// LANES k_grouped_down's sums, bit for bit: four chains of blocks 4k, 4k + 1, ...,
// products rounded before they are added, the chains as (0 + 1) + (2 + 3). Its
// 48 registers more leave three waves a SIMD, and a layer of 11 to 63 tokens of
// the Gemma shape takes 0.8 to 1.8 us longer (uniform routing 16 tokens 85.8 us
// against 84.9, 63 tokens 120.3 against 118.5).
// Four waves of about 94 registers per workgroup, several to a CU, so that one's
// staging runs under another's dots (8 waves 64 us against 57 at 512 tokens;
// two batches ahead instead of one 58.5). Before, one workgroup walked all of
// an expert's tokens, rereading the weights for each 16: 512 tokens of the
// Gemma shape 104 us, 173 zipf-skewed 93, 64 tokens 47; now 57, 31 and 33
// (143 MB of weights, 4.4 TB/s).
template <int NKB, int NW, bool LANES, bool REC, bool SCAN>
__global__ __launch_bounds__(NW * 64, LANES ? 3 : 4) void k_mfma_down_tok(
    const uint8_t* __restrict__ bank, int64_t expert_bytes, int64_t gu_bytes, const int32_t* __restrict__ meta,
    const uint32_t* __restrict__ tiles, const int32_t* __restrict__ plist, const uint8_t* __restrict__ q8m, int P,
    float* ydn, int H, int I, int E, int32_t* rec, const uint32_t* __restrict__ trec) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int NTH = NW * 64, NC = LANES ? 4 : 1, NBUF = 2;
    const int nbj = I >> 5, dn_tile = nbj * 288, RG = H / 64, JG = (RG + NW - 1) / NW;
    const int n_units = (int)(tiles[0] >> 18) * JG, per = (n_units + 7) >> 3, ur = (int)blockIdx.x >> 3;
    const int unit = ((int)blockIdx.x & 7) * per + ur;  // as k_mfma_gu_tok's
    if (ur >= per || unit >= n_units) return;
    int e, q0 = 0, nt;
    const uint16_t* tp = nullptr;  // SCAN: the tile's pairs, which are also their positions in q8m
    if constexpr (SCAN) {
        const uint32_t* tr = trec + unit / JG * TREC;
        e = (int)(tr[0] & 0xFFFF);
        nt = (int)(tr[0] >> 16);
        tp = reinterpret_cast<const uint16_t*>(tr + 1);
    } else {
        const uint32_t v0 = tiles[unit / JG];
        const int g = (int)(v0 >> 8) & 1023, c0 = (int)(v0 & 255) * MT;
        e = meta[1 + g];
        q0 = meta[1 + E + g] + c0;
        nt = min(MT, meta[1 + 2 * E + g] - c0);
    }
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, li = t & 15, lg = lane >> 4;
    const int qt = SCAN ? (int)tp[li] : q0 + min(li, nt - 1);  // slot li's position (past the tile: the last token's, never written out)
    const int rw0 = (unit % JG) * NW + wave, rg = min(rw0, RG - 1);  // this wave's 64 rows
    // LDS: the tokens' act words [nbj][4][MT] (g, g+4) | [nbj][MT] d | the waves' scales [4][nbj][16] f16
    uint2* xq = reinterpret_cast<uint2*>(lds);
    float* xd = reinterpret_cast<float*>(lds + (size_t)nbj * 512);
    uint8_t* scl = lds + (size_t)nbj * 576 + (size_t)wave * nbj * 128;
    const __amdgpu_buffer_rsrc_t rw =
        buf_rsrc(bank + (int64_t)e * expert_bytes + gu_bytes + (int64_t)rg * 4 * dn_tile, (uint32_t)(4 * dn_tile));
    u32x4 ss[4], aw[NBUF][4];
#pragma unroll
    for (int m = 0; m < 4; ++m)
        ss[m] = __builtin_amdgcn_raw_buffer_load_b128(rw, min(lane * 16, nbj * 32 - 16), m * dn_tile, 0);
    auto load = [&](int kb, int buf) __attribute__((always_inline)) {  // lane group g: block 4*kb + g of row li of each tile
        const uint32_t vo = nbj * 32 + min(4 * kb + lg, nbj - 1) * 256 + li * 16;
#pragma unroll
        for (int m = 0; m < 4; ++m) aw[buf][m] = __builtin_amdgcn_raw_buffer_load_b128(rw, vo, m * dn_tile, 0);
    };
#pragma unroll
    for (int k = 0; k < NBUF - 1; ++k) load(k, k);
    {
        constexpr int R = (4 * NKB * 64 + NTH - 1) / NTH, RD = (4 * NKB * 16 + NTH - 1) / NTH;
        const uint2* q2 = reinterpret_cast<const uint2*>(q8m);
        uint2 w[R];
        float dv[RD];
#pragma unroll
        for (int r = 0; r < R; ++r) {  // item i: slot i % 16 = li, as NTH is a multiple of 16
            const int i = r * NTH + t;
            if (i < nbj * 64) w[r] = q2[(int64_t)(i >> 4) * P + qt];
        }
#pragma unroll
        for (int r = 0; r < RD; ++r) {
            const int i = r * NTH + t;
            if (i < nbj * 16) dv[r] = __uint_as_float(q2[(int64_t)P * nbj * 4 + (int64_t)(i >> 4) * P + qt].x);
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (r * NTH + t < nbj * 64) xq[r * NTH + t] = w[r];
#pragma unroll
        for (int r = 0; r < RD; ++r)
            if (r * NTH + t < nbj * 16) xd[r * NTH + t] = dv[r];
    }
#pragma unroll
    for (int m = 0; m < 4; ++m)
        if (lane * 16 < nbj * 32) *reinterpret_cast<u32x4*>(scl + m * nbj * 32 + lane * 16) = ss[m];
    __syncthreads();
    if (rw0 >= RG) return;
    float acc[NC][4][4];
#pragma unroll
    for (int i = 0; i < NC * 16; ++i) acc[i >> 4][i >> 2 & 3][i & 3] = 0.0f;
    const int p = SCAN ? qt : plist[qt];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
        if (kb + NBUF - 1 < NKB) load(kb + NBUF - 1, (kb + NBUF - 1) % NBUF);
        uint32_t w[4][4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const u32x4 v = aw[kb % NBUF][m];
            w[m][0] = v.x;
            w[m][1] = v.y;
            w[m][2] = v.z;
            w[m][3] = v.w;
            quad_transpose(w[m][0], w[m][1], w[m][2], w[m][3]);
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int blk = kb * 4 + b;
            if (blk < nbj) {  // uniform
                const uint2 q = xq[(blk * 4 + lg) * MT + li];
                const float ad = xd[blk * MT + li];
                const long bop = (long)(((uint64_t)q.y << 32) | q.x);
                const v4i c8 = start_sums(bop);
                v4i d[4];
                v4f sp[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const float dw = h2f(*reinterpret_cast<const uint16_t*>(scl + (m * nbj + blk) * 32 + lg * 8 + (li & 3) * 2));
                    sp[m] = scale_products(dw, ad);
                }
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    d[m] = __builtin_amdgcn_mfma_i32_16x16x32_i8(nib_op(w[m][b]), bop, c8, 0, 0, 0);
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    if constexpr (REC) {  // test record: the (row, token) blocks' int32 dots
                        if (li < nt)
#pragma unroll
                            for (int v = 0; v < 4; ++v)
                                rec[((int64_t)p * H + rg * 64 + m * 16 + 4 * lg + v) * nbj + blk] = d[m][v];
                    }
                    float(&a)[4] = acc[b % NC][m];
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        a[v] = LANES ? a[v] + (float)d[m][v] * sp[m][v] : fmaf((float)d[m][v], sp[m][v], a[v]);
                    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]));
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // one block's MFMA results live at a time
        }
    }
    if (li < nt) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            float y[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                y[v] = acc[0][m][v];
                if constexpr (LANES) y[v] = (y[v] + acc[1][m][v]) + (acc[2][m][v] + acc[3][m][v]);
            }
            *reinterpret_cast<float4*>(ydn + (int64_t)p * H + rg * 64 + m * 16 + 4 * lg) =
                make_float4(y[0], y[1], y[2], y[3]);
        }
    }
}

// Down rows of over 32 blocks of active expert g for its tokens, 16 at a time.
// The workgroup takes RT consecutive 16-row down tiles (they share each
// block's activation operand); wave w works on K slice w (blocks [w*BW,
// w*BW+BW) below nbj); the slice partials of a (row, token) are summed in
// slice order into y[pair][row]. The partials overlay the tiles' scales in LDS
// (restaged for each 16 tokens), so two workgroups fit a CU. Blocks go in
// batches of four, NBUF batches in flight (register buffers). ONCE: the rows are
// loaded past the caches (nontemporal).
template <int BW, int RT, int NBUF, bool REC, bool ONCE>
__global__ __launch_bounds__(GT, 4) void k_mfma_down(const uint8_t* bank, int64_t expert_bytes, int64_t gu_bytes,
                                                     const int32_t* meta, const int32_t* plist, const uint8_t* q8m,
                                                     int P, float* ydn, int H, int I, int E, int32_t* rec) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int nbj = I >> 5, dn_tile = nbj * 288;
    const int u = blockIdx.x, g = blockIdx.y;
    if (g >= meta[1 + 3 * E]) return;
    const int e = meta[1 + g], s0 = meta[1 + E + g], n = meta[1 + 2 * E + g];
    // LDS: the tiles' scales [RT][nbj][16] f16; slice partials [GW][RT][16][MT]
    // in the same bytes once the K loop is done
    uint16_t* scl = reinterpret_cast<uint16_t*>(lds);
    float* red = reinterpret_cast<float*>(lds);
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), li = t & 15, lg = (t >> 4) & 3;
    const int bs = wave * BW;
    const int tile0 = u * RT;
    const uint8_t* D0 = bank + (int64_t)e * expert_bytes + gu_bytes;  // the expert's down tiles
    // the RT tiles: qs of tile tile0+m at m*dn_tile + nbj*32 from D0 + tile0*dn_tile
    const __amdgpu_buffer_rsrc_t rw = buf_rsrc(D0 + (int64_t)tile0 * dn_tile, (uint32_t)(RT * dn_tile));
    const __amdgpu_buffer_rsrc_t ra = buf_rsrc(q8m, (uint32_t)P * nbj * Q8_BLK);  // < NO_TOKEN bytes
    constexpr int NBB = 4, NBATCH = BW / NBB;
    // this slice's batches (uniform; none when the slice starts past nbj)
    const int nbat = max(0, min(NBATCH, (nbj - bs + NBB - 1) / NBB));
    // this lane's row and block in a batch, and in the slice's last one
    const uint32_t vw4 = nbj * 32 + lg * 256 + li * 16;
    const uint32_t vwl = nbj * 32 + min(lg, nbj - 1 - (bs + (nbat - 1) * NBB)) * 256 + li * 16;
    for (int c0 = 0; c0 < n; c0 += MT) {
        const int nt = min(MT, n - c0);
        const int q = s0 + c0 + min(li, nt - 1), p = plist[q];
        // this lane's operand words of block bb: 8 bytes at bb * 32P + vq (the
        // 16 tokens' words of a lane group in 128 contiguous bytes), d and
        // qsum at P * nbj * 32 + bb * 8P + vd
        const bool ok = li < nt;
        const uint32_t vq = ok ? (uint32_t)(lg * P + q) * 8 : NO_TOKEN;
        const uint32_t vd = ok ? (uint32_t)P * nbj * 32 + (uint32_t)q * 8 : NO_TOKEN;
        // blocks in batches of four, the loads of the batch NBUF - 1 ahead
        // issued before the current batch's MFMAs (NBUF register buffers)
        uint32_t aw[NBUF][NBB][RT];
        ActOp av[NBUF][NBB];
        // one 16-byte load per tile for the batch's four blocks,
        // lane group g taking all four qs words of its row in block 4k+g (1 KB
        // contiguous per wave), turned into word g of each block by
        // quad_transpose when the batch is consumed (past the slice its last
        // batch again, past the row its last block, never used: no read leans on
        // the descriptor's range check, which may not see the scalar offset)
        auto load = [&](int k, int buf) __attribute__((always_inline)) {
            const int kw = min(k, nbat - 1);  // uniform
            const uint32_t vw = kw < nbat - 1 ? vw4 : vwl;
#pragma unroll
            for (int m = 0; m < RT; ++m) {
                const u32x4 v =
                    __builtin_amdgcn_raw_buffer_load_b128(rw, vw, m * dn_tile + (bs + kw * NBB) * 256, ONCE ? 2 : 0);
                aw[buf][0][m] = v.x;
                aw[buf][1][m] = v.y;
                aw[buf][2][m] = v.z;
                aw[buf][3][m] = v.w;
            }
#pragma unroll
            for (int b = 0; b < NBB; ++b) {
                const int bb = min(bs + k * NBB + b, nbj - 1);
                av[buf][b] = act_op_m(ra, vq, vd, bb * 32 * P, bb * 8 * P);
            }
        };
        float acc[RT][4];
#pragma unroll
        for (int m = 0; m < RT; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[m][v] = 0.0f;
#pragma unroll
        for (int k = 0; k < NBUF - 1; ++k)
            if (k < nbat) load(k, k);
        stage<8>(  // the tiles' scales to LDS, with the first batches in flight
            RT * nbj * 8,
            [&](int i) {
                const int k = i / (nbj * 8), r = i - k * nbj * 8;
                return reinterpret_cast<const uint32_t*>(D0 + (int64_t)(tile0 + k) * dn_tile)[r];
            },
            [&](int i, uint32_t v) { reinterpret_cast<uint32_t*>(scl)[i] = v; });
        __syncthreads();
        // rounds of NBUF batches, register buffer j holding batch kb + j; the
        // rounds are a loop (not unrolled), so a block's offsets are scalar
        // adds rather than registers held across the slice
#pragma unroll 1
        for (int kb = 0; kb < nbat; kb += NBUF) {
#pragma unroll
          for (int j = 0; j < NBUF; ++j) {
            const int k = kb + j;
            if (k >= nbat) break;  // uniform
            // unconditional (past the slice: the last block again), so the
            // wait below counts only this batch's loads, not the prefetch's
            load(k + NBUF - 1, (j + NBUF - 1) % NBUF);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < RT; ++m) quad_transpose(aw[j][0][m], aw[j][1][m], aw[j][2][m], aw[j][3][m]);
#pragma unroll
            for (int b = 0; b < NBB; ++b) {
                if (bs + k * NBB + b < nbj) {  // uniform
                    const ActOp a = av[j][b];
                    const v4i c = c_init(a.qsum);
#pragma unroll
                    for (int m = 0; m < RT; ++m) {
                        const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(nib_op(aw[j][b][m]), a.b, c, 0, 0, 0);
                        if constexpr (REC) {  // test record: D = the (row, token) blocks' int32 dots
                            if (li < nt)
#pragma unroll
                                for (int v = 0; v < 4; ++v)
                                    rec[((int64_t)p * H + (tile0 + m) * 16 + 4 * lg + v) * nbj + bs + k * NBB + b] = d[v];
                        }
                        float sc[4];
                        scales4(scl + (m * nbj + bs + k * NBB + b) * 16 + 4 * lg, sc);
#pragma unroll
                        for (int v = 0; v < 4; ++v) acc[m][v] = fmaf((float)d[v], sc[v] * a.d, acc[m][v]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);  // one block's MFMA results live at a time
            }
          }
        }
        __syncthreads();  // every wave is done with the scales
#pragma unroll
        for (int m = 0; m < RT; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[((wave * RT + m) * 16 + 4 * lg + v) * MT + li] = acc[m][v];
        __syncthreads();
        for (int i = t; i < RT * 16 * nt; i += GT) {  // (tile, row, token) sums over the slices in order
            const int m = i / (16 * nt), r = (i / nt) % 16, tt = i % nt;
            float sv = 0.0f;
#pragma unroll
            for (int q = 0; q < GW; ++q) sv = sv + red[((q * RT + m) * 16 + r) * MT + tt];
            ydn[(int64_t)plist[s0 + c0 + tt] * H + (tile0 + m) * 16 + r] = sv;
        }
        __syncthreads();
    }
}

// The MFMA groups' act quants from q8m back into the pairs' rows of q8a
// ([P][nbj][40]), for the debug copy: MFMA group blockIdx.y, one thread per
// (position, block, word) of the group.
__global__ __launch_bounds__(256) void k_q8m_rows(const uint32_t* q8m, const int32_t* meta, const int32_t* plist,
                                                  uint8_t* q8a, int P, int nbj, int E) {
    const int g = blockIdx.y;
    if (g >= meta[1 + 3 * E]) return;  // not an MFMA group
    const int s0 = meta[1 + E + g], n = meta[1 + 2 * E + g];
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n * nbj * 10; i += gridDim.x * 256) {
        const int wd = i % 10, j = i / 10 % nbj, q = s0 + i / (10 * nbj), wq = wd - 2;
        const int64_t o = wd < 2 ? ((int64_t)P * nbj * 4 + (int64_t)j * P + q) * 2 + wd
                                 : (((int64_t)j * 4 + (wq & 3)) * P + q) * 2 + (wq >> 2);
        reinterpret_cast<uint32_t*>(q8a + ((int64_t)plist[q] * nbj + j) * Q8_BLK)[wd] = q8m[o];
    }
}

// x_out[t] = x[t] + sum_k (y[t*K+k] * w[t*K+k]), slots in order
// (ft-model/src/lib.rs:1634-1646).
__global__ __launch_bounds__(256) void k_grouped_combine(const float* y, const float* wts, const float* x, float* out,
                                                         int H, int K) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, s = blockIdx.y;
    if (i >= H) return;
    const float xv = x[(int64_t)s * H + i];
    float h = 0.0f;
    for (int k0 = 0; k0 < K; k0 += 8) {  // the loads of 8 slots issued together, then the sum in slot order
        float yv[8], wv[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int k = min(k0 + q, K - 1);
            yv[q] = y[((int64_t)s * K + k) * H + i];
            wv[q] = wts[s * K + k];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float part = yv[q] * wv[q];
            h = k0 + q < K ? h + part : h;
        }
    }
    out[(int64_t)s * H + i] = xv + h;
}

int check_grouped_shape(const char* nm, int64_t B, int64_t H, int64_t I, int64_t E, int64_t K) {
    if (H != 2816 && H != 4096)
        return fail(FT_HIP_E_SHAPE, "%s: hidden=%lld: built for hidden 2816 and 4096", nm, (long long)H);
    if (I <= 0 || I % 32 || I / 32 > 512)
        return fail(FT_HIP_E_SHAPE, "%s: inter=%lld must be a multiple of 32 in [32, 16384]", nm, (long long)I);
    if (E <= 0 || E > 1024) return fail(FT_HIP_E_SHAPE, "%s: n_experts not in [1, 1024]", nm);
    if (K <= 0 || K > 32 || K > E) return fail(FT_HIP_E_SHAPE, "%s: top_k not in [1, min(32, n_experts)]", nm);
    if (B < 0 || B * K > MAX_PAIRS) return fail(FT_HIP_E_SHAPE, "%s: n_seqs*top_k must be <= %d", nm, MAX_PAIRS);
    return FT_HIP_OK;
}

}  // namespace

extern "C" size_t ft_hip_moe_layer_grouped_workspace_bytes(int64_t n_seqs, int64_t hidden, int64_t inter,
                                                           int64_t n_experts, int64_t top_k) {
    // by division, so that no product below can wrap
    if (n_seqs < 0 || top_k <= 0 || top_k > 1024 || n_seqs > 65535 / top_k || hidden <= 0 || hidden > 32 * 4096 ||
        inter <= 0 || inter > 32 * 4096 || n_experts <= 0 || n_experts > 65535)
        return 0;
    return group_ws(nullptr, n_seqs, hidden, inter, n_experts, top_k).bytes;
}

extern "C" int ft_hip_moe_layer_grouped(ft_hip_ctx* ctx, void* stream, const float* x, float* x_out, int64_t n_seqs,
                                        int64_t hidden, int64_t inter, int64_t n_experts, int64_t top_k,
                                        const float* router_w, const float* router_bias, const float* expert_scale,
                                        const void* bank, int32_t* ids, float* wts, void* workspace,
                                        size_t workspace_bytes, float* dbg_gu, void* dbg_act) {
    clear_error();
    const char* nm = "moe_layer_grouped";
    if (int rc = check_grouped_shape(nm, n_seqs, hidden, inter, n_experts, top_k)) return rc;
    const GroupWs w = group_ws(workspace, n_seqs, hidden, inter, n_experts, top_k);
    if (workspace_bytes < w.bytes) return fail(FT_HIP_E_SHAPE, "%s: workspace_bytes=%zu < %zu", nm, workspace_bytes, w.bytes);
    if (!ctx || !x || !x_out || !router_w || !bank || !ids || !wts || !workspace)
        return fail(FT_HIP_E_INVALID, "%s: null argument", nm);
    if (reinterpret_cast<uintptr_t>(bank) & 15) return fail(FT_HIP_E_SHAPE, "%s: bank must be 16-byte aligned", nm);
    if (n_seqs == 0) return FT_HIP_OK;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int H = (int)hidden, I = (int)inter, E = (int)n_experts, K = (int)top_k;
    const int P = (int)(n_seqs * top_k), nb = H / 32, nbj = I / 32;
    const int64_t eb = ft_hip_fused_expert_bytes(hidden, inter);
    const int64_t gu_bytes = 2LL * I * nb * 18;
    int rc;
    const float* inv = ctx->input_norm ? w.inv : nullptr;
    const bool parts = ft::route_parts_fits(hidden, n_experts, top_k, n_seqs);
    if (parts) {  // the whole routing; its group sums in ydn, which the down launch writes after their last reader
        if ((rc = ft::launch_route_topk(stream, router_w, x, router_bias, expert_scale, ctx->input_norm, w.inv, w.q8x,
                                        w.ydn, ids, wts, hidden, n_experts, top_k, n_seqs)))
            return rc;
    } else if (n_experts * 16 >= hidden / 32) {  // logits, norm scale and q8(x) in one launch
        if ((rc = ft::launch_route_prep(stream, router_w, x, router_bias, ctx->input_norm, w.inv, w.q8x, w.logits,
                                        hidden, n_experts, n_seqs)))
            return rc;
    } else {
        if (inv && (rc = ft::launch_rms_inv(stream, x, w.inv, hidden, n_seqs))) return rc;
        if ((rc = ft::launch_router_logits(stream, router_w, x, router_bias, inv, w.logits, hidden, n_experts, n_seqs)))
            return rc;
        if ((rc = ft_hip_quantize_q8(ctx, stream, x, hidden, w.q8x, hidden, n_seqs))) return rc;
    }
    // the routing inside the grouping launch for few experts (up to 32, in up
    // to 4 rounds of 1024/E tokens), else its own launch: one workgroup
    // ranking 128 logits per token is LDS-bound (batch 16 of the Gemma
    // shape: 188.4 vs 172.6 us/token); at 8 experts it saves the launch
    const bool topk_in = !parts && E <= 32 && n_seqs <= 4 * (1024 / E);
    if (!topk_in && !parts && (rc = ft_hip_topk_router(ctx, stream, w.logits, expert_scale, ids, wts, n_experts, top_k, n_seqs)))
        return rc;
    // groups of >= n_mfma tokens take the MFMA tile kernels, the others the
    // dot4 kernels; rows longer than 32 blocks (I > 1024) only the former.
    // Automatic (0): every group on one family, MFMA from 2/3 of a pair per
    // expert on (layers of the Gemma shape with uniform / zipf-skewed routing, MFMA
    // against dot4: 8 tokens 65 / 48 us against 60 / 48, 11 tokens 71 / 54 against 73 /
    // 60, 16 tokens 82 / 52 against 87 / 83, 24 tokens 101 / 60 against 103 / 111, 63
    // tokens 119 / 86 against 160 / 252: dot4's cost grows with an expert's tokens),
    // and, below 4, only from 64 pairs (H 2816) or 96 (H 4096) on: fewer leave the
    // MFMA kernels' larger units too few (32 experts of I 704: 48 pairs 50 / 47 against
    // 47 / 54, 64 pairs 50 / 48 against 52 / 62; 32 experts of H 4096, I 1024, K-split
    // form: 48 pairs 85 / 72 against 77 / 74, 64 88 / 76 against 86 / 88, 96 90 / 84
    // against 101 / 111); from 40 in layers of up to two units of the K-split gate|up
    // per CU (16 experts of I 704: 48 pairs 40 / 39 against 45 / 51; 32 experts, 748
    // units, 40 pairs 48 against 44)
    int n_mfma = ctx->grouped_mfma_min;
    const bool sparse = P < 4LL * n_experts;
    // (tile, act block) units of the MFMA gate|up with every group on it, at most
    const int64_t all_units = (int64_t)nbj * std::min(P, P / MT + std::min(E, P));
    if (n_mfma <= 0) {
        const int few = all_units <= 2 * 256 ? 40 : H == 2816 ? 64 : 96;
        n_mfma = sparse && (3LL * P < 2 * n_experts || P < few) ? std::numeric_limits<int>::max() : 1;
    }
    if (nbj > 32) n_mfma = 1;
    // Automatic, below 4 pairs per expert: the down sums in the dot4 kernels' order, so that where the line above
    // lies in this range shows in no output bit (another order of 22 block sums moves q8 quants of the layers that
    // follow: 3e-4 of the state after four layers). From there on, and where the caller splits the experts, one chain
    // in block order, the faster form.
    const bool lanes = ctx->grouped_mfma_min <= 0 && sparse;
    // every expert on the dot4 kernels, routing already in ids: the dot4
    // workgroups find their expert's pairs themselves (no grouping launch)
    const bool scan = !topk_in && n_mfma > P && P <= SCAN_MAX;
    const bool rec = ctx->rec_gu && ctx->rec_dn;
    // Every expert on the token-tile MFMA kernels: up to TILE_SCAN pairs their waves find the tiles themselves, which
    // costs them less than the grouping launch: 16 tokens of the Gemma shape with uniform / zipf-skewed routing 82.3 /
    // 55.4 us a layer against 85.9 / 59.5, 20 tokens 97.2 / 60.9 against 100.2 / 64.5, 63 tokens 119.4 / 85.8 against
    // 121.7 / 86.7, 64 tokens as much.
    const bool tscan = !topk_in && n_mfma == 1 && P <= TILE_SCAN && E <= 256 && nbj <= 32 && !rec && !dbg_act;
    if (!scan && !tscan) {
        hipLaunchKernelGGL(topk_in ? k_group_pairs<true> : k_group_pairs<false>, dim3(1), dim3(1024), 0, s,
                           (const int32_t*)ids, P, E, n_mfma, w.meta, w.plist, w.ppos, (const float*)w.logits,
                           expert_scale, ids, wts, K);
        if ((rc = launch_status("moe_layer_grouped/group"))) return rc;
    }
    const int gmax = std::min(E, P);
    const int gbig = std::min(gmax, n_mfma > P ? 0 : P / n_mfma);  // at most this many groups of >= n_mfma tokens
    const bool dot4 = n_mfma > 1, mfma = n_seqs >= n_mfma;
    const int n_tiles = std::min(P, P / MT + gbig);  // at most this many token tiles
    if (mfma && (int64_t)P * nbj * Q8_BLK >= (int64_t)NO_TOKEN)
        return fail(FT_HIP_E_SHAPE, "%s: %d pairs x %d act blocks: the MFMA path's activation buffer must stay under 2 GiB",
                    nm, P, nbj);
    // a block-dot record (ft_hip_set_block_dot_record, tests only) selects
    // the instantiations that store every int32 block dot
    int32_t* rgu = ctx->rec_gu;
    int32_t* rdn = ctx->rec_dn;
    if (dot4) {
        const size_t lds_gu = (size_t)NT * nb * 40 + sizeof(float) * (GW * NT * 64 + NT * 64 + NT * 32) + 4 * NT * 10;
        auto kern = scan ? (H == 2816 ? (rec ? k_grouped_gu<11, true, true> : k_grouped_gu<11, false, true>)
                                      : (rec ? k_grouped_gu<16, true, true> : k_grouped_gu<16, false, true>))
                         : (H == 2816 ? (rec ? k_grouped_gu<11, true, false> : k_grouped_gu<11, false, false>)
                                      : (rec ? k_grouped_gu<16, true, false> : k_grouped_gu<16, false, false>));
        hipLaunchKernelGGL(kern, dim3(nbj, gmax), dim3(GT), lds_gu, s, (const uint8_t*)bank, eb,
                           (const int32_t*)w.meta, (const int32_t*)w.plist, (const uint8_t*)w.q8x, w.q8a, dbg_gu, inv, H,
                           I, E, K, n_mfma, rgu, (const int32_t*)ids, P);
        if ((rc = launch_status("moe_layer_grouped/gate_up"))) return rc;
    }
    if (mfma) {
        auto gate_up = [&](auto kern, int nw, int kh, int jpw) {
            const size_t lds_mg = (size_t)nb / kh * ((MT * 8 + 2) * 4 + MT * 4) + (size_t)nw * nb / 8 * 128;
            hipLaunchKernelGGL(kern, dim3(((nbj + jpw - 1) / jpw * n_tiles + 7) / 8 * 8), dim3(nw * 64), lds_mg, s,
                               (const uint8_t*)bank, eb, (const int32_t*)w.meta, (uint32_t*)w.ppos,
                               (const int32_t*)w.plist, (const uint8_t*)w.q8x, w.q8m, dbg_gu, inv, I, E, K, P, rgu,
                               (const int32_t*)ids, (uint32_t*)w.q8a);
        };
        // Forms of one kernel. H 2816. Few tokens per expert: the weights bound it (one tile per expert, 285 MB
        // for all 128 of the Gemma shape), and small workgroups that hold half of the tokens' rows at a time
        // (31 KB of LDS; their 165 registers let 3 on a CU) spread them best over the CUs: 64 tokens 63 us against 73 for the other
        // form, 127 tokens 64 against 73 (zipf-skewed 55 against 65). More tokens: the VALU bounds it, and 8
        // waves share one staging of whole rows, two workgroups to a CU: 512 tokens 118-126 us against 137,
        // 173 zipf-skewed tokens 67 against 70; at 10 pairs per expert 74 against 80 (zipf-skewed 67, 71).
        // Few (tile, act block) units for the chip's 256 CUs: a wave that walks whole rows takes 25 us (H 2816) or
        // 35 to 80 (H 4096, 4 to 16 waves a CU) however few they are, so the 8 slices of a row go to 8 waves. Layers,
        // that form against the other, uniform / zipf-skewed routing, by this bound on the units: H 2816 (I 704) 550
        // units 43 / 43 us against 58 / 59, 704 (under 9 pairs per expert) 42 / 39 against 47 / 46, 792 53 / 42 against
        // 50 / 48, 902 58 / 56 against 55 / 56, 1056 (over) 64 / 64 against 67 / 67, 1760 94 / 95 against 80 / 81; H
        // 4096 (I 1024) 512 53 against 62, 704 58 / 61 against 61 / 63, 768 72 against 69, 1024 80 against 71.
        // H 4096 has two forms more, by the units too: the 4 waves with half of the rows spread few units over more
        // CUs, the 16 of one CU read the rows in larger pieces (the large-expert shape): 1312 units 70 / 73 us
        // against 114, 2624 115 / 103 against 137 / 132, 3072 124 / 128 against 142 / 139, 3584 148 / 141 against 143
        // / 139, 4032 186 / 180 against 167 / 160.
        const int64_t units = (int64_t)nbj * n_tiles;
        const bool ks = !rec && units <= (H == 2816 && P >= 9 * E ? 4 : 3) * 256;
        if (H == 2816 && ks)
            gate_up(tscan ? k_mfma_gu_tok<11, 8, 4, 6, 1, false, true, true>
                          : k_mfma_gu_tok<11, 8, 4, 6, 1, false, false, true>, 8, 1, 1);
        else if (ks)
            gate_up(tscan ? k_mfma_gu_tok<16, 8, 2, 16, 1, false, true, true>
                          : k_mfma_gu_tok<16, 8, 2, 16, 1, false, false, true>, 8, 1, 1);
        else if (H == 2816 && P < 9 * E)
            gate_up(tscan ? k_mfma_gu_tok<11, 4, 3, 5, 2, false, true, false>
                    : rec ? k_mfma_gu_tok<11, 4, 3, 8, 2, true, false, false>
                          : k_mfma_gu_tok<11, 4, 3, 5, 2, false, false, false>, 4, 2, 4);
        else if (H == 2816)
            gate_up(tscan ? k_mfma_gu_tok<11, 8, 4, 6, 1, false, true, false>
                    : rec ? k_mfma_gu_tok<11, 8, 4, 6, 1, true, false, false>
                          : k_mfma_gu_tok<11, 8, 4, 6, 1, false, false, false>, 8, 1, 8);
        else if (!rec && units <= 12 * 256)
            gate_up(tscan ? k_mfma_gu_tok<16, 4, 3, 5, 2, false, true, false>
                          : k_mfma_gu_tok<16, 4, 3, 5, 2, false, false, false>, 4, 2, 4);
        else
            gate_up(tscan ? k_mfma_gu_tok<16, 16, 4, 6, 1, false, true, false>
                    : rec ? k_mfma_gu_tok<16, 16, 4, 6, 1, true, false, false>
                          : k_mfma_gu_tok<16, 16, 4, 6, 1, false, false, false>, 16, 1, 16);
        if ((rc = launch_status("moe_layer_grouped/gate_up_mfma"))) return rc;
        if (dbg_act) {  // the debug copy below reads q8a's pair rows
            hipLaunchKernelGGL(k_q8m_rows, dim3(64, (unsigned)gbig), dim3(256), 0, s,
                               (const uint32_t*)w.q8m, (const int32_t*)w.meta, (const int32_t*)w.plist, w.q8a, P, nbj,
                               E);
            if ((rc = launch_status("moe_layer_grouped/q8m_rows"))) return rc;
        }
    }
    if (dbg_act && hipMemcpyAsync(dbg_act, w.q8a, (size_t)P * nbj * Q8_BLK, hipMemcpyDeviceToDevice, s) != hipSuccess)
        return fail(FT_HIP_E_LAUNCH, "%s: debug copy failed", nm);
    if (dot4) {
        const size_t lds_dn = (size_t)NTD * nbj * 40;
        auto kern = scan ? (nbj <= 24 ? (rec ? k_grouped_down<6, true, true> : k_grouped_down<6, false, true>)
                                      : (rec ? k_grouped_down<8, true, true> : k_grouped_down<8, false, true>))
                         : (nbj <= 24 ? (rec ? k_grouped_down<6, true, false> : k_grouped_down<6, false, false>)
                                      : (rec ? k_grouped_down<8, true, false> : k_grouped_down<8, false, false>));
        hipLaunchKernelGGL(kern, dim3(H / DU, gmax), dim3(GT), lds_dn, s, (const uint8_t*)bank, eb, gu_bytes,
                           (const int32_t*)w.meta, (const int32_t*)w.plist, (const uint8_t*)w.q8a, w.ydn, H, I, E,
                           n_mfma, rdn, (const int32_t*)ids, P);
        if ((rc = launch_status("moe_layer_grouped/down"))) return rc;
    }
    if (mfma) {
        if (nbj <= 32) {
            constexpr int NW = 4;
            const size_t lds_md = (size_t)nbj * (576 + NW * 128);
            auto form = [&](auto ln, auto rc, auto sn) {
                constexpr bool LN = decltype(ln)::value, RC = decltype(rc)::value, SN = decltype(sn)::value;
                return nbj <= 24 ? k_mfma_down_tok<6, NW, LN, RC, SN> : k_mfma_down_tok<8, NW, LN, RC, SN>;
            };
            constexpr std::true_type T{};
            constexpr std::false_type F{};
            auto pick = [&](auto ln) { return tscan ? form(ln, F, T) : rec ? form(ln, T, F) : form(ln, F, F); };
            auto kern = lanes ? pick(T) : pick(F);
            hipLaunchKernelGGL(kern, dim3(((H / 64 + NW - 1) / NW * n_tiles + 7) / 8 * 8), dim3(NW * 64), lds_md, s,
                               (const uint8_t*)bank, eb, gu_bytes, (const int32_t*)w.meta, (const uint32_t*)w.ppos,
                               (const int32_t*)w.plist, (const uint8_t*)w.q8m, P, w.ydn, H, I, E, rdn,
                               (const uint32_t*)w.q8a);
        } else {  // long rows: DRT tiles per workgroup, 8 K slices of 56 (rows up to 448 blocks) or 64 blocks
            constexpr int DRT = 4;
            const size_t lds_md = std::max((size_t)DRT * nbj * 32, sizeof(float) * GW * DRT * 16 * MT);
            // The rows go past the caches while an expert's tokens mostly fit one tile of 16: past it they are read
            // again (layer of the large-expert shape, 8 experts, past / through: 16 tokens 171.5 / 174.0 us, 32 178.6 /
            // 180.5, 40 179.6 / 181.5, 48 234.5 / 236.6, 56 295 / 294, 64 296.8 / 295.5, 96 330.7 / 322.6).
            const bool once = !rec && P <= 12 * E;
            auto form = [&](auto on, auto rc) {
                constexpr bool ON = decltype(on)::value, RC = decltype(rc)::value;
                return nbj <= 8 * 56 ? k_mfma_down<56, DRT, 2, RC, ON> : k_mfma_down<64, DRT, 2, RC, ON>;
            };
            auto kern = once ? form(std::true_type{}, std::false_type{})
                        : rec ? form(std::false_type{}, std::true_type{})
                              : form(std::false_type{}, std::false_type{});
            hipLaunchKernelGGL(kern, dim3(H / (16 * DRT), gbig), dim3(GT), lds_md, s, (const uint8_t*)bank, eb,
                               gu_bytes, (const int32_t*)w.meta, (const int32_t*)w.plist, (const uint8_t*)w.q8m, P,
                               w.ydn, H, I, E, rdn);
        }
        if ((rc = launch_status("moe_layer_grouped/down_mfma"))) return rc;
    }
    hipLaunchKernelGGL(k_grouped_combine, dim3((H + 255) / 256, (unsigned)n_seqs), dim3(256), 0, s, (const float*)w.ydn,
                       (const float*)wts, x, x_out, H, K);
    return launch_status("moe_layer_grouped/combine");
}

// ---------------------------------------------------------------------------
// The L-layer stack for a batch (forward_batch's expert section for every
// layer, ft-model/src/lib.rs:1507-1606, called per layer from :1151-1154).
// Workspace: the layer workspace for max_seqs, then two [max_seqs][H] f32
// states and [L][max_seqs*K] ids/wts for callers that pass no record.
// ---------------------------------------------------------------------------
namespace {
struct StackWs {
    void* layer;
    size_t layer_bytes;
    float* state[2];
    int32_t* ids;
    float* wts;
    size_t bytes;
};

StackWs stack_ws(void* base, int64_t max_seqs, int64_t H, int64_t I, int64_t E, int64_t K, int64_t L) {
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    StackWs w{};
    uint8_t* p = (uint8_t*)base;
    size_t off = 0;
    w.layer = p;
    w.layer_bytes = group_ws(nullptr, max_seqs, H, I, E, K).bytes;
    off += up(w.layer_bytes);
    for (int i = 0; i < 2; ++i) {
        w.state[i] = (float*)(p + off);
        off += up(sizeof(float) * max_seqs * H);
    }
    w.ids = (int32_t*)(p + off);
    off += up(sizeof(int32_t) * L * max_seqs * K);
    w.wts = (float*)(p + off);
    off += up(sizeof(float) * L * max_seqs * K);
    w.bytes = off;
    return w;
}
}  // namespace

extern "C" size_t ft_hip_moe_stack_grouped_workspace_bytes(int64_t max_seqs, int64_t hidden, int64_t inter,
                                                           int64_t n_experts, int64_t top_k, int64_t n_layers) {
    if (max_seqs < 0 || hidden <= 0 || inter <= 0 || n_experts <= 0 || top_k <= 0 || n_layers <= 0) return 0;
    return stack_ws(nullptr, max_seqs, hidden, inter, n_experts, top_k, n_layers).bytes;
}

extern "C" int ft_hip_moe_stack_grouped(ft_hip_ctx* ctx, void* stream, const float* x_in, float* x_out,
                                        int64_t n_seqs, int64_t max_seqs, int64_t hidden, int64_t inter,
                                        int64_t n_experts, int64_t top_k, int64_t n_layers, const void* banks,
                                        const float* routers, const float* router_bias, const float* expert_scale,
                                        int32_t* ids, float* wts, void* workspace, size_t workspace_bytes) {
    clear_error();
    const char* nm = "moe_stack_grouped";
    if (int rc = check_grouped_shape(nm, max_seqs, hidden, inter, n_experts, top_k)) return rc;
    if (n_seqs < 0 || n_seqs > max_seqs)
        return fail(FT_HIP_E_SHAPE, "%s: n_seqs=%lld not in [0, max_seqs=%lld]", nm, (long long)n_seqs, (long long)max_seqs);
    if (n_layers <= 0) return fail(FT_HIP_E_SHAPE, "%s: n_layers=%lld must be positive", nm, (long long)n_layers);
    if (!ctx || !x_in || !x_out || !banks || !routers || !workspace) return fail(FT_HIP_E_INVALID, "%s: null argument", nm);
    if ((ids == nullptr) != (wts == nullptr)) return fail(FT_HIP_E_INVALID, "%s: give ids and wts or neither", nm);
    const StackWs w = stack_ws(workspace, max_seqs, hidden, inter, n_experts, top_k, n_layers);
    if (workspace_bytes < w.bytes)
        return fail(FT_HIP_E_SHAPE, "%s: workspace_bytes=%zu < %zu (for max_seqs %lld)", nm, workspace_bytes, w.bytes,
                    (long long)max_seqs);
    if (n_seqs == 0) return FT_HIP_OK;
    const int64_t eb = ft_hip_fused_expert_bytes(hidden, inter);
    const int64_t P = n_seqs * top_k;
    const size_t lbytes = group_ws(nullptr, n_seqs, hidden, inter, n_experts, top_k).bytes;
    const float* src = x_in;
    for (int64_t l = 0; l < n_layers; ++l) {
        // the last layer writes x_out, unless it would overwrite its own input
        // in a one-layer in-place call
        const bool last = l == n_layers - 1;
        float* dst = last && !(n_layers == 1 && x_out == x_in) ? x_out : w.state[l & 1];
        int32_t* il = ids ? ids + l * P : w.ids + l * P;
        float* wl = wts ? wts + l * P : w.wts + l * P;
        const uint8_t* bank = static_cast<const uint8_t*>(banks) + l * n_experts * eb;
        if (int rc = ft_hip_moe_layer_grouped(ctx, stream, src, dst, n_seqs, hidden, inter, n_experts, top_k,
                                              routers + l * n_experts * hidden,
                                              router_bias ? router_bias + l * n_experts : nullptr,
                                              expert_scale ? expert_scale + l * n_experts : nullptr, bank, il, wl,
                                              w.layer, lbytes, nullptr, nullptr))
            return rc;
        src = dst;
    }
    if (src != x_out) {
        hipError_t e = hipMemcpyAsync(x_out, src, sizeof(float) * n_seqs * hidden, hipMemcpyDeviceToDevice,
                                      reinterpret_cast<hipStream_t>(stream));
        if (e != hipSuccess) return fail(FT_HIP_E_LAUNCH, "%s: copy of the result: %s", nm, hipGetErrorString(e));
    }
    return FT_HIP_OK;
}
