"""Where the one-token kernels read: their source compiled for the CPU, run lane by lane over weights, scales and rows that end at an
unmapped page.  Only addresses are checked (a workgroup's threads run one after the other, so the sums are meaningless); a read past
the last row of the last expert, or before the first, ends the program with the case that made it.  No GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "machx_inference_engine_amd", "csrc")

# stand-ins for what the host compiler lacks; lane exchanges return the lane's own value
SHIM = r"""
#include <hip/hip_runtime.h>
#include <math.h>
#include <signal.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include <sys/mman.h>
#include <unistd.h>
#undef __global__
#undef __device__
#undef __host__
#undef __shared__
#undef __forceinline__
#undef __align__
#undef __launch_bounds__
#define __global__
#define __device__
#define __host__
#define __shared__
#define __forceinline__ inline
#define __align__(n) __attribute__((aligned(n)))
#define __launch_bounds__(...)
struct Idx { uint32_t x, y, z; };
static Idx threadIdx, blockIdx, blockDim, gridDim;
static inline void __syncthreads() {}
template <class T> static inline T __shfl_xor(T v, int) { return v; }
typedef _Float16 shim_h2 __attribute__((ext_vector_type(2)));
static inline uint32_t shim_u(uint32_t a, uint32_t) { return a; }
static inline shim_h2 shim_fp4(uint32_t, float, int) { return shim_h2{}; }
static inline float shim_dot(shim_h2, shim_h2, float c, bool) { return c; }
#define __expf expf
#define __builtin_amdgcn_perm(a, b, c) shim_u(a, b)
#define __builtin_amdgcn_sdot4(a, b, c, d) ((c) + (a))
#define __builtin_amdgcn_update_dpp(o, v, a, b, c, d) (v)
#define __builtin_amdgcn_ds_bpermute(i, v) (v)
#define __builtin_amdgcn_mbcnt_lo(m, v) (v)
#define __builtin_amdgcn_mbcnt_hi(m, v) (threadIdx.x & 63u)
#define __builtin_amdgcn_sched_barrier(x)
#define __builtin_amdgcn_cvt_scalef32_pk_f16_fp4 shim_fp4
#define __builtin_amdgcn_fdot2 shim_dot
"""

CHECK = r"""
namespace mxq { alignas(64) uint8_t lds[1u << 20]; }
using namespace mxq;
static char what[256];
static void on_fault(int) { const char* m = "read outside its buffer: "; write(1, m, strlen(m)); write(1, what, strlen(what)); _exit(3); }
// n bytes that end where an unmapped page starts; another one lies in front
static uint8_t* guarded(size_t n) {
    const size_t page = 4096, up = (n + page - 1) / page * page;
    uint8_t* p = static_cast<uint8_t*>(mmap(nullptr, up + 2 * page, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    mprotect(p + page, up, PROT_READ | PROT_WRITE);
    return p + page + up - n;
}
struct Held { uint8_t* p; size_t n; Held(size_t bytes) : p(guarded(bytes)), n(bytes) {}
    ~Held() { const size_t up = (n + 4095) / 4096 * 4096; munmap(p + n - up - 4096, up + 8192); } };
template <class Fn> static void run(uint32_t threads, uint32_t gx, uint32_t gy, Fn fn) {
    blockDim = {threads, 1, 1};
    gridDim = {gx, gy, 1};
    for (uint32_t y = 0; y < gy; ++y)
        for (uint32_t b = 0; b < gx; ++b)
            for (uint32_t t = 0; t < threads; ++t) { blockIdx = {b, y, 0}; threadIdx = {t, 0, 0}; fn(); }
}
static uint32_t tile_k(uint32_t K) { return (K + 255) / 256 * 256; }
"""

MOE = r"""
constexpr uint32_t E = 2;
template <class F, int NW, int G, int EPI> static void experts(const char* name, uint32_t K, const typename F::Bank& bank, uint32_t N, uint32_t f16) {
    constexpr int R = 1, U = 2;
    Held q8(K / 32 * 40), h16(2 * K), out(2 * N), bias(4 * E * N), w(2);
    int32_t id = (int32_t)E - 1;
    MoeArgs a{};
    a.xq8 = q8.p; a.act_f16 = f16 ? reinterpret_cast<const half_t*>(h16.p) : nullptr; a.topk_idx = &id; a.out = reinterpret_cast<half_t*>(out.p);
    a.bias0 = a.bias1 = reinterpret_cast<const float*>(bias.p); a.route_w = reinterpret_cast<const half_t*>(w.p);
    a.act_div = 1; a.K = K; a.N = N; a.KT = tile_k(K); a.n_experts = E;
    snprintf(what, sizeof what, "moe_gemv_kernel %s, %d matrices, K = %u, %d lanes per row\n", name, NW, K, G);
    run(kGemvThreads, 1, 1, [&] { moe_gemv_kernel<F, 1, NW, R, G, U, EPI>(bank, bank, a); });
}
template <int G> static void all(uint32_t K) {
    const uint32_t N = 4 * (64 / G) + 1;   // one full round of row groups and a ragged one
    for (uint32_t f16 = 0; f16 < 2; ++f16) {
        {
            Held qs((size_t)E * N * K / 2), e((size_t)E * N * K / 32);
            const FmtMxfp4Soa::Bank b{qs.p, e.p, (uint64_t)N * K / 2, (uint64_t)N * K / 32, K};
            experts<FmtMxfp4Soa, 1, G, EPI_DOWN_BIAS>("mxfp4", K, b, N, f16);
            experts<FmtMxfp4Soa, 2, G, EPI_OAI>("mxfp4", K, b, N, f16);
        }
        Held qs((size_t)E * N * K), d((size_t)E * N * K / 16);
        const FmtQ8Soa::Bank b{reinterpret_cast<const int8_t*>(qs.p), reinterpret_cast<const uint16_t*>(d.p), (uint64_t)N * K, (uint64_t)N * K / 32, K};
        experts<FmtQ8Soa, 1, G, EPI_DOWN_WEIGHTED>("q8_0", K, b, N, f16);
        experts<FmtQ8Soa, 2, G, EPI_SILU>("q8_0", K, b, N, f16);
    }
}
int main() {
    signal(SIGSEGV, on_fault);
    signal(SIGBUS, on_fault);
    for (uint32_t K = 32; K <= 4352; K += K % 128 ? 32 : K < 1024 ? 32 : 128) { all<16>(K); all<32>(K); all<64>(K); }
    return 0;
}
"""

DENSE = r"""
template <class F, int G> static void plain(const char* name, uint32_t K, const typename F::W& w, uint32_t N) {
    Held q8(K / 32 * 40), y(2 * N);
    const GemvSeg<F, half_t> s{w, reinterpret_cast<half_t*>(y.p), nullptr};
    const uint32_t KT = tile_k(K), units = (K + 63) / 64;
    snprintf(what, sizeof what, "gemv_q8_kernel %s, K = %u, %d lanes per row\n", name, K, G);
    if (K % F::K_ALIGN) return;
    run(kGemvThreads, 2, 1, [&] { gemv_q8_kernel<F, 1, 1, G, 2, half_t>(s, s, q8.p, K, N, KT, 1, 0); });
    snprintf(what, sizeof what, "gemv_q8_deep_kernel %s, K = %u, %d lanes per row\n", name, K, G);
    run(kGemvThreads, 2, 1, [&] { gemv_q8_deep_kernel<F, G, half_t>(s, q8.p, K, N, KT, 0); });
    if (G != 64) return;
    snprintf(what, sizeof what, "gemv_q8_wide_kernel %s, K = %u\n", name, K);
    run(kGemvThreads, 2, 1, [&] { gemv_q8_wide_kernel<F, 1, 1, half_t>(s, s, q8.p, K, N, KT, 1, 0); });
    snprintf(what, sizeof what, "gemv_q8_wide_pair_kernel %s, K = %u\n", name, K);
    if (K % 64 == 0 && units % 32 == 0 && units < 256) run(2 * units, 2, 1, [&] { gemv_q8_wide_pair_kernel<F, half_t>(s, q8.p, K, N, KT, 0); });
}
template <int G> static void all(uint32_t K) {
    const uint32_t N = 8 * (64 / G) + 1;
    {
        Held qs((size_t)N * K / 2), e((size_t)N * K / 32);
        plain<FmtMxfp4Soa, G>("mxfp4", K, FmtMxfp4Soa::W{qs.p, e.p, K}, N);
    }
    {
        Held qs((size_t)N * K), d((size_t)N * K / 16);
        const FmtQ8Soa::W w{reinterpret_cast<const int8_t*>(qs.p), reinterpret_cast<const uint16_t*>(d.p), K};
        plain<FmtQ8Soa, G>("q8_0 planes", K, w, N);
        plain<FmtQ8SoaW, G>("q8_0 planes, interleaved", K, w, N);
    }
    {
        Held b((size_t)N * K / 32 * 34);
        plain<FmtQ8Aos, G>("q8_0 blocks", K, FmtQ8Aos::W{b.p, K / 32 * 34}, N);
    }
    if (K % 256) return;
    {
        Held b((size_t)N * K / 256 * 144);
        plain<FmtQ4K, G>("q4_K", K, FmtQ4K::W{b.p, K / 256 * 144}, N);
    }
    Held b((size_t)N * K / 256 * 210);
    plain<FmtQ6K, G>("q6_K", K, FmtQ6K::W{b.p, K / 256 * 210}, N);
}
int main() {
    signal(SIGSEGV, on_fault);
    signal(SIGBUS, on_fault);
    for (uint32_t K : {32u, 64u, 96u, 512u, 736u, 768u, 1024u, 1120u, 1152u, 2048u, 2880u, 3072u, 4096u, 4608u, 8192u, 10240u, 14336u}) { all<16>(K); all<32>(K); all<64>(K); }
    return 0;
}
"""


def kernels(name, before):
    """The part of a source file in front of the section comment `before`, which holds the kernels and nothing of the host side."""
    text = open(os.path.join(CSRC, name)).read()
    assert text.count(before) == 1
    return text.split(before)[0].replace('#include "mxq_mmq.h"', "") + "}  // namespace mxq\n"


@pytest.mark.parametrize("name,before,program", [
    ("moe.hip", "// ---------------------------------------------------------------- fp16-activation decode", MOE),
    ("gemv.hip", "// true if the launch was made: one matrix, one token", DENSE)], ids=["experts", "dense"])
def test_reads_stay_inside_the_weights(tmp_path, name, before, program):
    # -O0: a load whose value the stand-ins drop is made all the same
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SHIM + kernels(name, before) + CHECK + program)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-std=c++17", "-O0", "-w", "-I", CSRC,
                    "-I", "/opt/rocm/include", str(src), "-o", str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout + p.stderr
