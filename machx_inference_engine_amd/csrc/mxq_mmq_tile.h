// Body of the loop over token tiles of mmq_kernel (mxq_mmq.h), for a tile of at most 2 TR rows from row t0 on; included there twice, as text (mmq_tile
// says why), so without a guard.  What it takes from around it: the template parameters P, TR, NW, WR, WK, EPI and NATIVE; the arguments a, lds, e
// (expert), t0, r_end (end of the expert's rows), kzi, G0, G1 (the workgroup's K range and its groups); lane, j, h, wave, wk, wr, wm; w (the wave's
// matrix), nb, n_rb (blocks of 32 elements, row blocks), gp (groups staged at once), single (all at once), q8_row_bytes, red (the exchange area).
const uint32_t nt = r_end - t0 < 2 * TR ? r_end - t0 : 2 * TR;
auto xrow = [&](uint32_t t) { return a.xq8 + (size_t)(t0 + t) * q8_row_bytes; };
auto hrow = [&](uint32_t t) { return a.act_f16 + (size_t)(t0 + t) * a.K; };
// token rows past the tile re-read its last row (their results are dropped)
const uint32_t jt = NATIVE ? (j & 15u) : j, row_a = jt < nt ? jt : nt - 1u;
typename std::conditional<NATIVE, MmqWalkNative<P, TR>, MmqWalk<P, TR, mmq_two_tails<P, TR, EPI>()>>::type walk;
MmqAct act{};
bool staged = false, requested = false;
// what the epilogue reads from global memory is requested ahead of the weight walk: a load issued in the epilogue
// would have to wait for the whole queue of weight words requested for the next row block before it
float rw[EPI == MMQ_DOWN_WEIGHTED ? TR : 1];
if constexpr (EPI == MMQ_DOWN_WEIGHTED) {
#pragma unroll
    for (int v = 0; v < TR; ++v) {
        const uint32_t t = mmq_row(v) + 4u * h;
        rw[v] = (float)a.route_w[t0 + (t < nt ? t : nt - 1u)];
    }
}
for (uint32_t rb = blockIdx.x; rb < n_rb; rb += gridDim.x) {
    const uint32_t n0 = (rb * WR + wr) * 32u;
    const uint32_t n = n0 + j < a.N ? n0 + j : a.N - 1u;
    // MMQ_OAI: the bias of this wave's matrix joins its partial sum before the exchange (wave wk = 0 of each matrix);
    // MMQ_DOWN_BIAS: added after the fp16 rounding of the sum, in the epilogue
    float bias_a = 0.f;
    if (EPI == MMQ_OAI || EPI == MMQ_DOWN_BIAS) {
        const float* bp = (NW == 2 && wm) ? a.bias1 : a.bias0;
        if (bp) bias_a = bp[(size_t)e * a.N + n];
    }
    float acc[TR];
#pragma unroll
    for (int v = 0; v < TR; ++v) acc[v] = 0.f;
    for (uint32_t gb = G0; gb < G1; gb += gp) {
        const uint32_t ge = gb + gp < G1 ? gb + gp : G1;          // groups [gb, ge) of this pass
        const uint32_t per = (ge - gb + WK - 1u) / WK;
        const uint32_t g_lo = gb + wk * per < ge ? gb + wk * per : ge, g_hi = g_lo + per < ge ? g_lo + per : ge;
        // the pipeline takes whole groups and a partial last group follows it, except where the producer loads both alike
        const uint32_t g_full = (NATIVE || g_hi < nb / 8u) ? g_hi : nb / 8u;
        if (!requested && g_lo < g_full) walk.prefetch(w, n, g_lo, g_full, h, nb);
        requested = false;
        if (!staged) {
            mmq_lds_barrier();                                        // the image of the previous pass is no longer read
            act = a.act_f16 ? mmq_stage_f16<TR, P::HAS_MIN, NATIVE>(lds, hrow, nt, gb * 256u, (ge - gb) * 256u, a.K)
                            : mmq_stage<TR, P::HAS_MIN, NATIVE>(lds, xrow, nt, gb * 256u, (ge - gb) * 256u, a.K, a.q8_split != 0);
            mmq_lds_barrier();
            staged = single;
        }
        const uint32_t a_off = row_a * act.stride + 16u * h + (NATIVE ? 64u * (j >> 4) : 0u);
        if (g_lo < g_full) walk.run(w, n, g_lo, g_full, gb, h, nb, act, a_off, acc);
        if (g_hi > g_full && g_lo <= g_full) walk.tail(w, n, g_full, gb, h, nb, act, a_off, acc);
        // the epilogue's operands are made to arrive here, while nothing else is outstanding: otherwise the wait for
        // them would sit in the epilogue, behind the weight words requested just below
        asm volatile("" : "+v"(bias_a));
        if constexpr (EPI == MMQ_DOWN_WEIGHTED) {
#pragma unroll
            for (int v = 0; v < TR; ++v) asm volatile("" : "+v"(rw[v]));
        }
        if (EPI == MMQ_OAI && ge == G1 && wk == 0) {
#pragma unroll
            for (int v = 0; v < TR; ++v) acc[v] += bias_a;
        }
        if (single && rb + gridDim.x < n_rb && g_lo < g_full) {
            // the next row block's first weight words, requested before the partial sums of this one meet
            const uint32_t nn0 = ((rb + gridDim.x) * WR + wr) * 32u;
            walk.prefetch(w, nn0 + j < a.N ? nn0 + j : a.N - 1u, g_lo, g_full, h, nb);
            requested = true;
        }
    }
    // ---- partial sums of the WK waves (and the NW matrices) meet in LDS; a workgroup of row blocks only has none to meet
    if constexpr (NW * WK > 1) {
        mmq_lds_barrier();
#pragma unroll
        for (int v = 0; v < TR; ++v) red[((size_t)wave * TR + v) * 64u + lane] = acc[v];
        mmq_lds_barrier();
    }
    if (wk == 0 && wm == 0) {
        // Row v of a lane is t0 + 4 h + mmq_row(v): the lane's share of an address is one 32-bit offset and the rest is
        // uniform.  The offset is made opaque here, once per row block: 2 TR addresses kept in registers across the
        // weight walk were what made the walk spill (Q6_K, TR = 16: 256 registers and 46 more in scratch).
        uint32_t lane_at = 4u * h * a.N + j;
        asm volatile("" : "+v"(lane_at));
        const bool col_ok = n0 + j < a.N;
        if (a.part) {
            float* base = a.part + ((size_t)kzi * a.M + t0) * a.N + n0;
#pragma unroll
            for (int v = 0; v < TR; ++v) {
                float s0 = acc[v];
                if constexpr (NW * WK > 1) {
                    s0 = 0.f;
#pragma unroll
                    for (int k = 0; k < WK; ++k) s0 += red[((size_t)(wr * WK + k) * TR + v) * 64u + lane];
                }
                if (mmq_row(v) + 4u * h < nt && col_ok) (base + (size_t)mmq_row(v) * a.N)[lane_at] = s0;
            }
        } else {
            half_t* base = a.out + (size_t)t0 * a.N + n0;
#pragma unroll
            for (int v = 0; v < TR; ++v) {
                float s0 = acc[v], s1 = 0.f;
                if constexpr (NW * WK > 1) {
                    s0 = 0.f;
#pragma unroll
                    for (int k = 0; k < WK; ++k) {
                        s0 += red[((size_t)((0 * WR + wr) * WK + k) * TR + v) * 64u + lane];
                        if (NW == 2) s1 += red[((size_t)((1 * WR + wr) * WK + k) * TR + v) * 64u + lane];
                    }
                }
                float o;
                if constexpr (EPI == MMQ_SILU) {
                    o = mmq_silu_mul(s0, s1);                                          // src/ops/moe_q8.cpp:94-97
                } else if constexpr (EPI == MMQ_OAI) {
                    // rounding points of the reference chain: half(acc + bias) per projection, then the fp16 activation
                    const float g = (float)(half_t)s0, u = (float)(half_t)s1;   // sums with their biases
                    o = mmq_swiglu_oai(g, u, a.alpha, a.limit);
                } else if constexpr (EPI == MMQ_DOWN_WEIGHTED) {
                    o = rw[v] * s0;                                                   // src/ops/moe_q8.cpp:143-144
                } else if constexpr (EPI == MMQ_DOWN_BIAS) {
                    o = (float)(half_t)s0;                                            // gemv out, then add_bias (elementwise.cpp:782-793)
                    if (a.bias0) o += bias_a;
                } else {
                    o = s0;
                }
                if (mmq_row(v) + 4u * h < nt && col_ok) (base + (size_t)mmq_row(v) * a.N)[lane_at] = (half_t)o;
            }
        }
    }
}
