// routing.hip — MoE routing and packing on the device, so that a layer never waits for the host
// between the router and the expert kernels:
//   router logits + softmax + top-k + renormalise + ascending-id order   src/ops/moe.cpp:22-216
//   softmax + top-k from logits already on the device                     src/ops/moe.cpp:366-412
//   packing arrays for one token                                          src/ops/moe.cpp:423-446
//   packing arrays for T tokens: stable counting sort by expert           src/model/qwen3moe_pack.cpp:5-31
#include "mxq_device.h"
#include "mxq_host.h"

namespace mxq {

// ---------------------------------------------------------------- router logits
// logit[t, e] = sum_h W_gate[e, h] * x[t, h], fp32 weights and sums.  One summation order for every call, whatever its batch,
// sizes and alignments, so that a token is routed alike alone, in a decode batch and in a prompt:
//   lane l takes the elements 4 l .. 4 l + 3 of every 256-element piece, router_dot4 over the four, pieces added in order;
//   the 64 lane sums meet in a balanced tree of neighbours.
// (32 products a lane at hidden 2048, then six levels: rms error against 64-bit sums 9.6e-8, maximum 5.4e-7, logits of unit variance.
// One fp32 MFMA accumulator per output, a chain of 128 or 256 products, takes 17 us where this takes 25 to 27 (2048 tokens, 128
// experts) but has rms 2.2e-7 to 2.9e-7 and maximum 1.8e-6: near ties are routed otherwise.)
__device__ __forceinline__ float router_dot4(const float4& w, const float (&x)[4]) {
    return __builtin_fmaf(w.w, x[3], __builtin_fmaf(w.z, x[2], __builtin_fmaf(w.x, x[0], w.y * x[1])));
}

// Halves N values per lane: the lane keeps the odd or the even ones (sel) and adds its partner's, or, with one value left, adds
// the partner's.  Level d pairs neighbouring groups of 2^d lanes.  DPP has no exchange at distance 4 or 8, but mirrors of 8 and 16
// lanes; `sel` of the lower levels is chosen so that mirrored lanes hold the same values.
template <int N, int D>
__device__ __forceinline__ void router_level(float (&v)[N], float (&o)[N > 1 ? N / 2 : 1], uint32_t lane) {
    auto partner = [](float x) {
        if constexpr (D == 0) return dpp_f<0xB1>(x);
        else if constexpr (D == 1) return dpp_f<0x4E>(x);
        else if constexpr (D == 2) return dpp_f<0x141>(x);
        else if constexpr (D == 3) return dpp_f<0x140>(x);
        else return __shfl_xor(x, 1 << D);
    };
    if constexpr (N == 1) {
        o[0] = v[0] + partner(v[0]);
    } else {
        const bool sel = ((D == 0 ? lane ^ (lane >> 2) : D == 1 ? (lane >> 1) ^ (lane >> 2) : D == 2 ? (lane >> 2) ^ (lane >> 3) : lane >> D) & 1u) != 0u;
#pragma unroll
        for (int i = 0; i < N / 2; ++i) {
            const float keep = sel ? v[2 * i + 1] : v[2 * i], send = sel ? v[2 * i] : v[2 * i + 1];
            o[i] = keep + partner(send);
        }
    }
}
template <int N, int D = 0>
__device__ __forceinline__ float router_tree(float (&v)[N], uint32_t lane) {
    float o[N > 1 ? N / 2 : 1];
    router_level<N, D>(v, o, lane);
    if constexpr (D == 5) return o[0];
    else return router_tree<(N > 1 ? N / 2 : 1), D + 1>(o, lane);
}

// One wave = MT tokens x NE experts, MT NE accumulators per lane (a power of two up to 64).  U: pieces whose loads are requested
// together.  The waves of a workgroup take neighbouring token tiles of the same experts.  Bound by: the load latency of a row at a
// few tokens, five vector instructions per four products at many (2048 tokens, 128 experts, hidden 2048: 17 us of issue, 25 to
// 27 measured; one wave per output, which reads W once per token: 140).
template <int MT, int NE, int U>
__global__ __launch_bounds__(256) void router_logits_kernel(const half_t* __restrict__ x, const float* __restrict__ W, float* __restrict__ logits, uint32_t T,
                                                            uint32_t hidden, uint32_t E) {
    constexpr int P = MT * NE;
    static_assert((P & (P - 1)) == 0 && P <= 64, "one result per lane at most");
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t tile = blockIdx.x * (blockDim.x / 64u) + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t t_tiles = (T + MT - 1u) / MT, e0 = tile / t_tiles * NE, t0 = tile % t_tiles * MT;
    if (e0 >= E) return;
    const uint2* xr[MT];
    const float4* wr[NE];
#pragma unroll
    for (int m = 0; m < MT; ++m) xr[m] = reinterpret_cast<const uint2*>(x + (size_t)(t0 + m < T ? t0 + m : T - 1u) * hidden);   // uniform; piece c: xr[64 c + lane]
#pragma unroll
    for (int n = 0; n < NE; ++n) wr[n] = reinterpret_cast<const float4*>(W + (size_t)(e0 + n < E ? e0 + n : E - 1u) * hidden);
    float acc[P];
#pragma unroll
    for (int p = 0; p < P; ++p) acc[p] = 0.f;
    struct Piece {
        uint2 x[MT];
        float4 w[NE];
    };
    auto load = [&](uint32_t c, Piece& p) {
#pragma unroll
        for (int n = 0; n < NE; ++n) p.w[n] = wr[n][64u * c + lane];
#pragma unroll
        for (int m = 0; m < MT; ++m) p.x[m] = xr[m][64u * c + lane];
    };
    auto add = [&](const Piece& p) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float v[4] = {h2f(p.x[m].x & 0xFFFFu), h2f(p.x[m].x >> 16), h2f(p.x[m].y & 0xFFFFu), h2f(p.x[m].y >> 16)};
#pragma unroll
            for (int n = 0; n < NE; ++n) acc[m * NE + n] += router_dot4(p.w[n], v);
        }
    };
    const uint32_t n_full = hidden / 256u;
    const bool last = n_full * 256u + lane * 4u < hidden;   // the lanes that take part in the last, partial piece
    Piece end{};
    if (P <= 4 && last) load(n_full, end);                  // few outputs: requested ahead of everything else
    for (uint32_t c = 0; c < n_full; c += U) {
        Piece p[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (U == 1 || c + u < n_full) load(c + u, p[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (U == 1 || c + u < n_full) add(p[u]);
    }
    if (last) {
        if (P > 4) load(n_full, end);
        add(end);
    }
    const float sum = router_tree(acc, lane);
    // which value this lane has kept: one bit per halving level, the level's `sel`
    const uint32_t key = ((lane ^ (lane >> 2)) & 1u) | (((lane >> 1) ^ (lane >> 2)) & 1u) << 1 | (((lane >> 2) ^ (lane >> 3)) & 1u) << 2 | (lane & 56u);
    const uint32_t k = key & (P - 1u), t = t0 + k / NE, e = e0 + k % NE;
    if (lane < P && t < T && e < E) logits[(size_t)t * E + e] = sum;
}

template <int MT, int NE, int U, uint32_t WV>
static int launch_router(hipStream_t st, const half_t* x, const float* W, float* logits, uint32_t T, uint32_t hidden, uint32_t E) {
    const uint32_t tiles = ((T + MT - 1u) / MT) * ((E + NE - 1u) / NE);
    hipLaunchKernelGGL((router_logits_kernel<MT, NE, U>), dim3((tiles + WV - 1u) / WV), dim3(64u * WV), 0, st, x, W, logits, T, hidden, E);
    return launch_status();
}
// The tile by the number of outputs: small tiles spread few outputs over the CUs, large ones read the rows less often.  Times with
// the top-k behind it, us, 1 x 1 (one wave per workgroup) / 2 x 2 / 4 x 4 / 8 x 8: 128 experts, hidden 2048: 16 tokens 6.8 / 6.9 / 7.9 /
// 13, 64 tokens 9.7 / 8.0 / 8.1 / 13, 333 tokens 26 / 16 / 11.9 / 13, 1024 tokens 67 / 35 / 21.5 / 18; 32 experts, hidden 2880:
// one token 4.8 / 6.2 / 7.5 / 14, 512 tokens 17 / 11 / 8.7 / 15, 2048 tokens 54 / 29 / 16.9 / 15.6.
static int launch_router_logits(hipStream_t st, const half_t* x, const float* W, float* logits, uint32_t T, uint32_t hidden, uint32_t E) {
    const uint32_t n = T * E;   // at most 65535 x 1024
    if (n <= 2048u) return launch_router<1, 1, 8, 1>(st, x, W, logits, T, hidden, E);
    if (n <= 8192u) return launch_router<2, 2, 4, 4>(st, x, W, logits, T, hidden, E);
    if (n < 65536u) return launch_router<4, 4, 1, 4>(st, x, W, logits, T, hidden, E);
    return launch_router<8, 8, 1, 4>(st, x, W, logits, T, hidden, E);
}

// ---------------------------------------------------------------- softmax + top-k
constexpr int kMaxTopK = 64;

__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d));
    return v;
}
// maximum over the wave in a scalar register: DPP inside the rows, row broadcasts across them, lane 63 holds the result
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    auto step = [&](uint32_t o) { v = o > v ? o : v; };
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// One wave per token, lane l holds the experts l, l + 64, .. (NJ of them).  p = softmax(logits); K rounds of a wave-wide
// maximum over the float bits of p (monotonic for p >= 0; 1 is added so that 0 can mark an expert that is taken), the
// highest id among exact ties; then every winner renormalises its own weight and finds its place by counting the winners
// with a lower id.  No barrier, no LDS: 2048 tokens of 128 experts, k = 8, take 3.8 us where one workgroup per token with
// two barriers per round and a serial sort took 11.8; one token of 32 experts 2.3 (4.4).
template <class LogitT, int NJ>
__global__ __launch_bounds__(256) void topk_kernel(const LogitT* logits, int32_t* topk_idx, half_t* topk_w, uint32_t E, uint32_t K, uint32_t n_tokens) {
    const uint32_t lane = threadIdx.x & 63u, t = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (t >= n_tokens) return;
    const LogitT* lg = logits + (size_t)t * E;
    float p[NJ];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const uint32_t e = lane + 64u * j;
        p[j] = e < E ? load_act(lg + e) : -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) m = fmaxf(m, p[j]);
    m = wave_max_f(m);
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        p[j] = lane + 64u * j < E ? __expf(p[j] - m) : 0.f;
        s += u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(group_sum<64>(p[j])), 63));
    }
    uint32_t key[NJ];
    unsigned long long taken[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        p[j] = p[j] / s;
        const uint32_t bits = f2u(p[j]) < 0xFFFFFFFEu ? f2u(p[j]) : 0xFFFFFFFEu;   // a NaN of all ones stays a key: every round has a winner
        key[j] = lane + 64u * j < E ? bits + 1u : 0u;
        taken[j] = 0ull;
    }
    float ren = 0.f;
    for (uint32_t kk = 0; kk < K; ++kk) {
        uint32_t best = key[0];
#pragma unroll
        for (int j = 1; j < NJ; ++j) best = key[j] > best ? key[j] : best;
        const uint32_t win = wave_max_u32(best);
        ren += u2f(win - 1u);
        bool open = true;
#pragma unroll
        for (int j = NJ - 1; j >= 0; --j) {
            const unsigned long long hit = open ? __ballot(key[j] == win && key[j] != 0u) : 0ull;
            if (hit) {
                const uint32_t l = 63u - (uint32_t)__builtin_clzll(hit);
                taken[j] |= 1ull << l;
                if (lane == l) key[j] = 0u;
                open = false;
            }
        }
    }
    const float inv = 1.0f / ren;
    uint32_t below = 0;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        if ((taken[j] >> lane) & 1ull) {
            const uint32_t at = below + (uint32_t)__builtin_popcountll(taken[j] & ((1ull << lane) - 1ull));
            topk_idx[(size_t)t * K + at] = (int32_t)(lane + 64u * j);
            float w = p[j] * inv;
            asm volatile("" : "+v"(w));   // an fp32 value first: the compiler would round the product to fp16 at once
            topk_w[(size_t)t * K + at] = (half_t)w;
        }
        below += (uint32_t)__builtin_popcountll(taken[j]);
    }
}

template <class LogitT>
static int launch_topk(hipStream_t st, const LogitT* logits, int32_t* topk_idx, half_t* topk_w, uint32_t E, uint32_t K, uint32_t n_tokens) {
    const dim3 grid((n_tokens + 3) / 4), block(256);
    if (E <= 64) hipLaunchKernelGGL((topk_kernel<LogitT, 1>), grid, block, 0, st, logits, topk_idx, topk_w, E, K, n_tokens);
    else if (E <= 128) hipLaunchKernelGGL((topk_kernel<LogitT, 2>), grid, block, 0, st, logits, topk_idx, topk_w, E, K, n_tokens);
    else if (E <= 256) hipLaunchKernelGGL((topk_kernel<LogitT, 4>), grid, block, 0, st, logits, topk_idx, topk_w, E, K, n_tokens);
    else hipLaunchKernelGGL((topk_kernel<LogitT, 16>), grid, block, 0, st, logits, topk_idx, topk_w, E, K, n_tokens);
    return launch_status();
}

// ---------------------------------------------------------------- packing
// One token (src/ops/moe.cpp:423-446): offsets by counting, identity order.
__global__ void pack_decode_kernel(const int32_t* topk_idx, const half_t* topk_w, uint32_t* expert_offsets, int32_t* sorted_idx, int32_t* tk_to_packed,
                                   half_t* weights_packed, uint32_t E, uint32_t K) {
    // thread e counts the slots routed below e
    for (uint32_t e = threadIdx.x; e <= E; e += blockDim.x) {
        uint32_t below = 0;
        for (uint32_t kk = 0; kk < K; ++kk) below += ((uint32_t)topk_idx[kk] < e) ? 1u : 0u;
        expert_offsets[e] = below;
    }
    for (uint32_t kk = threadIdx.x; kk < K; kk += blockDim.x) {
        sorted_idx[kk] = 0;
        tk_to_packed[kk] = (int32_t)kk;
        weights_packed[kk] = topk_w[kk];
    }
}

// T tokens: stable counting sort of the T*K slots by expert id, in one launch.  Workgroup g sorts the slots of the Q experts
// from e0 = Q g on: it reads all ids, its waves a contiguous range each, counts the slots of every one of its experts (a
// ballot each) and those of all experts below e0, which is where its own begin; the counts of the waves meet in LDS, and in a
// second round over its ids a lane whose slot is one of the workgroup's knows its place.  So nothing passes between workgroups, at the
// price of reading the ids E / Q times, from L2.  With at most R = 4 or 16 slots a lane the ids stay in registers
// between the rounds (R = 0: read again).  One expert a workgroup up to 128 experts (128 experts, 16384 slots 10.5 us on cold caches,
// four experts a workgroup 14.6), four beyond, where the ids would be read too often.  Bound by the vector instructions per 64 slots.  us, one
// workgroup that ranks the slots of all experts with a ballot per id bit (bound by the pipes of its one CU) / this: 32 experts, 128
// slots 4.7 / 4.0; 128 experts, 2664 slots 6.9 / 4.7, 16384 slots 17.4 / 7.4, 65536 slots 101 / 21; 256 experts, 16384 slots 18.7 / 10.9;
// 1024 experts, 256 slots 10.2 / 3.7, 36000 slots 72 / 16.
template <int R, uint32_t Q>
__global__ __launch_bounds__(1024) void pack_kernel(const int32_t* __restrict__ topk_idx, const uint16_t* __restrict__ topk_w, uint32_t n, uint32_t K, uint32_t E,
                                                    uint32_t* __restrict__ expert_offsets, int32_t* __restrict__ sorted_idx,
                                                    uint16_t* __restrict__ weights_packed, int32_t* __restrict__ tk_to_packed) {
    __shared__ uint32_t counts[16][Q + 1];   // [wave]: slots of the Q experts, slots of experts below
    const uint32_t tid = threadIdx.x, lane = tid & 63u, n_waves = blockDim.x / 64u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t e0 = blockIdx.x * Q, n_own = E - e0 < Q ? E - e0 : Q;
    const uint32_t batches = (n + 63u) / 64u, per = (batches + n_waves - 1u) / n_waves;   // of 64 slots; a wave's
    const uint64_t lo64 = (uint64_t)wave * per * 64u, hi64 = lo64 + (uint64_t)per * 64u;
    const uint32_t lo = lo64 < n ? (uint32_t)lo64 : n, hi = hi64 < n ? (uint32_t)hi64 : n;
    constexpr int U = R ? R : 4;
    uint32_t id[U];
    auto load = [&](uint32_t c) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = c + 64u * u + lane;
            id[u] = i < hi ? (uint32_t)topk_idx[i] : 0xFFFFFFFFu;   // no expert's: slots without an expert of the bank are left out
        }
    };
    uint32_t cnt[Q] = {}, below = 0;
    auto count = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            below += (uint32_t)__popcll(__ballot(id[u] < e0));
#pragma unroll
            for (uint32_t q = 0; q < Q; ++q) cnt[q] += (uint32_t)__popcll(__ballot(id[u] == e0 + q));
        }
    };
    if constexpr (R > 0) {
        load(lo);
        count();
    } else {
        for (uint32_t c = lo; c < hi; c += 64u * U) {
            load(c);
            count();
        }
    }
    if (lane <= Q) {
        uint32_t v = below;
#pragma unroll
        for (uint32_t q = 0; q < Q; ++q) v = lane == q ? cnt[q] : v;
        counts[wave][lane] = v;
    }
    __syncthreads();
    // lane q <= Q: the sum over all waves and the one over the waves before this one
    uint32_t all = 0, before = 0;
    for (uint32_t w = 0; w < n_waves; ++w) {
        const uint32_t v = lane <= Q ? counts[w][lane] : 0u;
        all += v;
        before += w < wave ? v : 0u;
    }
    uint32_t at[Q], first = (uint32_t)__builtin_amdgcn_readlane((int)all, (int)Q);
#pragma unroll
    for (uint32_t q = 0; q < Q; ++q) {
        if (tid == 0 && q < n_own) expert_offsets[e0 + q] = first;
        at[q] = first + (uint32_t)__builtin_amdgcn_readlane((int)before, (int)q);
        if (q < n_own) first += (uint32_t)__builtin_amdgcn_readlane((int)all, (int)q);
    }
    if (tid == 0 && e0 + n_own == E) expert_offsets[E] = first;
    const bool small = n <= 65536u;
    const uint32_t inv = K > 1u ? 0xFFFFFFFFu / K + 1u : 0u;   // slot / K by a multiplication: exact below 2^16
    auto place = [&](uint32_t c) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = c + 64u * u + lane, rel = id[u] - e0;
            if (__ballot(rel < n_own) == 0ull) continue;
            uint32_t p = 0;
#pragma unroll
            for (uint32_t q = 0; q < Q; ++q) {
                const unsigned long long m = __ballot(rel == q);
                const uint32_t r = at[q] + (uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                p = rel == q ? r : p;
                at[q] += (uint32_t)__popcll(m);
            }
            if (rel < n_own) {
                sorted_idx[p] = (int32_t)(K == 1u ? i : small ? __umulhi(i, inv) : i / K);
                weights_packed[p] = topk_w[i];
                tk_to_packed[i] = (int32_t)p;
            }
        }
    };
    if constexpr (R > 0) {
        place(lo);
    } else {
        for (uint32_t c = lo; c < hi; c += 64u * U) {
            load(c);
            place(c);
        }
    }
}

}  // namespace mxq

using namespace mxq;

extern "C" {

int mx_moe_topk_from_logits(mx_stream_t s, const uint16_t* logits, int32_t* topk_idx, uint16_t* topk_w, uint32_t E, uint32_t K, uint32_t n_tokens) {
    MX_REQUIRE_PTR(logits); MX_REQUIRE_PTR(topk_idx); MX_REQUIRE_PTR(topk_w);
    MX_REQUIRE_SHAPE(E > 0 && E <= 1024 && K > 0 && K <= E && K <= (uint32_t)kMaxTopK && n_tokens > 0);
    return launch_topk(as_stream(s), reinterpret_cast<const half_t*>(logits), topk_idx, reinterpret_cast<half_t*>(topk_w), E, K, n_tokens);
}

int mx_moe_router(mx_stream_t s, const uint16_t* x, const float* W_gate, int32_t* topk_idx, uint16_t* topk_w, uint32_t n_tokens, uint32_t hidden,
                  uint32_t n_experts, uint32_t k, float* logits_ws) {
    MX_REQUIRE_PTR(x); MX_REQUIRE_PTR(W_gate); MX_REQUIRE_PTR(topk_idx); MX_REQUIRE_PTR(topk_w); MX_REQUIRE_PTR(logits_ws);
    MX_REQUIRE_SHAPE(n_tokens > 0 && n_tokens <= 65535 && hidden > 0 && hidden % 4 == 0 && n_experts > 0 && n_experts <= 1024 && k > 0 && k <= n_experts &&
                     k <= (uint32_t)kMaxTopK);
    MX_REQUIRE_ALIGN(x, 8); MX_REQUIRE_ALIGN(W_gate, 16);
    hipStream_t st = as_stream(s);
    if (int rc = launch_router_logits(st, reinterpret_cast<const half_t*>(x), W_gate, logits_ws, n_tokens, hidden, n_experts)) return rc;
    return launch_topk(st, (const float*)logits_ws, topk_idx, reinterpret_cast<half_t*>(topk_w), n_experts, k, n_tokens);
}

int mx_moe_build_pack_decode(mx_stream_t s, const int32_t* topk_idx, const uint16_t* topk_w, uint32_t* expert_offsets, int32_t* sorted_idx,
                             int32_t* tk_to_packed, uint16_t* weights_packed, uint32_t E, uint32_t K) {
    MX_REQUIRE_PTR(topk_idx); MX_REQUIRE_PTR(topk_w); MX_REQUIRE_PTR(expert_offsets); MX_REQUIRE_PTR(sorted_idx); MX_REQUIRE_PTR(tk_to_packed);
    MX_REQUIRE_PTR(weights_packed);
    MX_REQUIRE_SHAPE(E > 0 && K > 0);
    hipLaunchKernelGGL(pack_decode_kernel, dim3(1), dim3(256), 0, as_stream(s), topk_idx, reinterpret_cast<const half_t*>(topk_w), expert_offsets, sorted_idx,
                       tk_to_packed, reinterpret_cast<half_t*>(weights_packed), E, K);
    return launch_status();
}

int mx_moe_build_packing_device(mx_stream_t s, const int32_t* topk_idx, const uint16_t* topk_w, uint32_t T, uint32_t K, uint32_t E, uint32_t* expert_offsets,
                                int32_t* sorted_idx, uint16_t* weights_packed, int32_t* tk_to_packed) {
    MX_REQUIRE_PTR(topk_idx); MX_REQUIRE_PTR(topk_w); MX_REQUIRE_PTR(expert_offsets); MX_REQUIRE_PTR(sorted_idx); MX_REQUIRE_PTR(tk_to_packed);
    MX_REQUIRE_PTR(weights_packed);
    MX_REQUIRE_SHAPE(E > 0 && E <= 65535 && K > 0 && T > 0 && (uint64_t)T * K <= 0x7FFFFFFFull);
    const uint32_t n = T * K, waves = n <= 256 ? 4u : n <= 2048 ? 8u : 16u, slots = (n + 64u * waves - 1u) / (64u * waves);   // a lane's
    hipStream_t st = as_stream(s);
#define MX_PACK(R, Q) \
    hipLaunchKernelGGL((pack_kernel<R, Q>), dim3((E + Q - 1u) / Q), dim3(64u * waves), 0, st, topk_idx, topk_w, n, K, E, expert_offsets, sorted_idx, weights_packed, tk_to_packed)
    if (E <= 128u) {
        if (slots <= 4u) MX_PACK(4, 1);
        else if (slots <= 16u) MX_PACK(16, 1);
        else MX_PACK(0, 1);
    } else {
        if (slots <= 4u) MX_PACK(4, 4);
        else if (slots <= 16u) MX_PACK(16, 4);
        else MX_PACK(0, 4);
    }
#undef MX_PACK
    return launch_status();
}

}  // extern "C"
