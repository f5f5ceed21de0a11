// MXFP4 x fp8 GEMM for the batches between the matvec and a prompt (17 to a few hundred rows) on
// gfx950: small output tiles over the whole GPU, each workgroup's waves splitting K.
//
// What bounds the 128 x 128 kernels there is the serial chain of k steps on the few CUs that their
// tiles reach: 4096 x 3584 at 96 rows is 32 tiles of 28 steps.  Here a workgroup owns one tile of
// 16 TN weight rows x 16 TM tokens, small enough that the launch fills the GPU in one round, and wave w
// of W takes a contiguous W-th of the k steps with the whole tile in its accumulators.  The waves
// share nothing while they run, so there is no barrier until their partial tiles, W of them, are
// added in wave order through the LDS.
//
// Every wave copies its own operands global -> LDS into a ring of D steps of its own (D - 1 in flight,
// counted vmcnt waits), although the MFMA takes them straight from registers: its layout puts
// adjacent lanes in different rows, and the memory path merges only adjacent lanes.  Measured on data
// in L2, 16 rows x 64 B per load instruction: 9 TB/s with the lane's row = lane % 16, 25-31 TB/s with
// its row = lane / 4 as the copies have it.  The same kernel with direct register loads took 10.5 us
// at 4096 x 3584 x 96 and 41 us at 3584 x 18944 x 96; this one takes 7.2 and 26.4, the 128 x 128
// kernel 20.9 and 109.4 (per-token activations, in a graph).
//
// Scale dwords are loaded into registers, four steps of a row (16 bytes) at a time.
#include "fp8kv_common.h"
#include "fp8kv_status.h"
#include "w4a8_common.h"

namespace fp8kv {
namespace w4a8_detail {

template <int TN, int TM>
struct SliceFrags {
    u32x4_t a[TN];
    v8i b[TM];
};

// Byte j of each of T scale dwords, tile i in byte i % 4 of word i / 4 (op_sel picks it).
template <int T>
__device__ __forceinline__ void pack_scales(const uint32_t (&s)[T], uint32_t (&out)[(T + 3) / 4], uint32_t sel)
{
#pragma unroll
    for (int g = 0; g < (T + 3) / 4; ++g) {
        const int n = T - 4 * g;
        const uint32_t s0 = s[4 * g], s1 = n > 1 ? s[4 * g + 1] : 0u;
        const uint32_t lo = __builtin_amdgcn_perm(s1, s0, sel);
        if (n <= 2) {
            out[g] = lo;
        } else {
            const uint32_t s2 = s[4 * g + 2], s3 = n > 3 ? s[4 * g + 3] : 0u;
            out[g] = (lo & 0xFFFFu) | (__builtin_amdgcn_perm(s3, s2, sel) << 16);
        }
    }
}

template <int TN, int TM, int... Is>
__device__ __forceinline__ void slice_mfmas(const SliceFrags<TN, TM>& f, const uint32_t (&sa)[(TN + 3) / 4],
                                            const uint32_t (&sb)[(TM + 3) / 4], f32x4_t (&acc)[TN][TM],
                                            std::integer_sequence<int, Is...>)
{
    ((acc[Is / TM][Is % TM] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
          (v8i){(int)f.a[Is / TM][0], (int)f.a[Is / TM][1], (int)f.a[Is / TM][2], (int)f.a[Is / TM][3], 0, 0, 0, 0},
          f.b[Is % TM], acc[Is / TM][Is % TM], 4, 0, (Is / TM) % 4, (int)sa[(Is / TM) / 4], (Is % TM) % 4,
          (int)sb[(Is % TM) / 4])), ...);
}

constexpr int kScaleSteps = 4;                       // steps whose scale dwords one load brings (16 bytes per row)

template <int TN, int TM, int W, int D>
struct SliceGeom {
    static constexpr int COPIES = TN + 2 * TM;         // 1 KB copies per wave and step
    static constexpr int WAVE_BYTES = 1024 * (D * COPIES > TN * TM ? D * COPIES : TN * TM);
    static constexpr int LDS = W * WAVE_BYTES;
    static_assert(D >= 2 && D <= 4 && (D - 1) * COPIES < 64 && LDS <= 160 * 1024, "ring");
};

template <int TN, int TM, int W, int D, bool TOK>
__global__ void __launch_bounds__(64 * W)
gemm_slice_kernel(Params P)
{
    using G = SliceGeom<TN, TM, W, D>;
    constexpr int BN = 16 * TN, BM = 16 * TM;
    extern __shared__ __align__(16) unsigned char smem[];
    int nb, mb;
    if (!tile_of(P, blockIdx.x, nb, mb)) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, j = lane >> 4;
    const int N0 = nb * BN, M0 = mb * BM;
    const int kh = P.K >> 1, ks = P.K >> 5;
    const int nsteps = P.K / kBK;
    const int s0 = nsteps * wave / W, s1 = nsteps * (wave + 1) / W;
    unsigned char* const ring = smem + wave * G::WAVE_BYTES;

    // copies: lane = row lane / 4, 16 bytes at 16 (lane % 4), so that four adjacent lanes read 64
    // contiguous bytes
    const uint8_t* const wtile = P.W + (int64_t)N0 * kh;
    const uint8_t* const xtile = P.Xq + (int64_t)M0 * P.K;
    uint32_t wo[TN], xo[TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
        wo[i] = (uint32_t)min(16 * i + (lane >> 2), P.N - 1 - N0) * (uint32_t)kh + 16u * (uint32_t)(lane & 3);
#pragma unroll
    for (int i = 0; i < TM; ++i)
        xo[i] = (uint32_t)min(16 * i + (lane >> 2), P.M - 1 - M0) * (uint32_t)P.K + 16u * (uint32_t)(lane & 3);
    auto issue = [&](int s) {
        unsigned char* slot = ring + ((s - s0) % D) * (1024 * G::COPIES);
        const uint8_t* wb = wtile + (int64_t)s * 64;
        const uint8_t* xb = xtile + (int64_t)s * 128;
#pragma unroll
        for (int i = 0; i < TN; ++i) dma16_to_lds(wb + wo[i], slot + 1024 * i);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            dma16_to_lds(xb + xo[i], slot + 1024 * (TN + 2 * i));
            dma16_to_lds(xb + 64 + xo[i], slot + 1024 * (TN + 2 * i + 1));
        }
    };
    // Scale dwords of steps s .. s + 3 of this lane's rows, in registers; those past the row's last step
    // belong to no wave, and the load stays inside the row.
    const uint8_t* const swtile = P.St + (int64_t)N0 * ks;
    const uint8_t* const sxtile = TOK ? swtile : P.Sx + (int64_t)M0 * ks;
    uint32_t so[TN], sxo[TM];
#pragma unroll
    for (int i = 0; i < TN; ++i) so[i] = (uint32_t)min(16 * i + r, P.N - 1 - N0) * (uint32_t)ks;
#pragma unroll
    for (int i = 0; i < TM; ++i) sxo[i] = (uint32_t)min(16 * i + r, P.M - 1 - M0) * (uint32_t)ks;
    struct Scales {
        u32x4_t w[TN];
        u32x4_t x[TOK ? 1 : TM];
    };
    auto load_scales = [&](Scales& q, int s) {
        typedef uint32_t dword4_t __attribute__((ext_vector_type(4), aligned(4)));
        const int c = min(s, nsteps - kScaleSteps), d = s - c;        // d uniform
        auto row = [&](const uint8_t* base, uint32_t off) {
            const u32x4_t v = *reinterpret_cast<const dword4_t*>(base + (int64_t)c * 4 + off);
            return d == 0 ? v : d == 1 ? (u32x4_t){v[1], v[2], v[3], v[3]}
                 : d == 2 ? (u32x4_t){v[2], v[3], v[3], v[3]} : (u32x4_t){v[3], v[3], v[3], v[3]};
        };
#pragma unroll
        for (int i = 0; i < TN; ++i) q.w[i] = row(swtile, so[i]);
        if constexpr (!TOK) {
#pragma unroll
            for (int i = 0; i < TM; ++i) q.x[i] = row(sxtile, sxo[i]);
        }
    };

    f32x4_t acc[TN][TM];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

    const uint32_t sel = (uint32_t)j | ((uint32_t)(j + 4) << 8);
    const int frag = r * 64 + 16 * j;
    if (s0 < s1) {
        Scales q;
        load_scales(q, s0);
#pragma unroll
        for (int b = 0; b < D - 1; ++b)
            if (s0 + b < s1) issue(s0 + b);
        for (int s = s0; s < s1; s += kScaleSteps) {
            Scales nxt = q;
#pragma unroll
            for (int t = 0; t < kScaleSteps; ++t) {
                const int st = s + t;
                if (st >= s1) break;
                // this wave's own copies of the step: those of up to D - 2 later steps may be in flight
                const int ahead = min(s1 - 1 - st, D - 2);
                if (D > 3 && ahead == 2) wait_vmcnt<2 * G::COPIES>();
                else if (D > 2 && ahead == 1) wait_vmcnt<G::COPIES>();
                else wait_vmcnt<0>();
                if (t == 0 && s + kScaleSteps < s1) load_scales(nxt, s + kScaleSteps);
                // the slot of step st - 1 was read into registers (lgkmcnt) before its MFMAs
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if (st + D - 1 < s1) issue(st + D - 1);
                const unsigned char* slot = ring + ((st - s0) % D) * (1024 * G::COPIES) + frag;
                SliceFrags<TN, TM> f;
#pragma unroll
                for (int i = 0; i < TN; ++i) f.a[i] = *reinterpret_cast<const u32x4_t*>(slot + 1024 * i);
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    f.b[i] = concat8(*reinterpret_cast<const u32x4_t*>(slot + 1024 * (TN + 2 * i)),
                                     *reinterpret_cast<const u32x4_t*>(slot + 1024 * (TN + 2 * i + 1)));
                uint32_t dw[TN], sa[(TN + 3) / 4], sb[(TM + 3) / 4];
#pragma unroll
                for (int i = 0; i < TN; ++i) dw[i] = q.w[i][t];
                pack_scales<TN>(dw, sa, sel);
                if constexpr (TOK) {
#pragma unroll
                    for (int g = 0; g < (TM + 3) / 4; ++g) sb[g] = 0x7F7F7F7Fu;
                } else {
                    uint32_t dx[TM];
#pragma unroll
                    for (int i = 0; i < TM; ++i) dx[i] = q.x[i][t];
                    pack_scales<TM>(dx, sb, sel);
                }
                slice_mfmas<TN, TM>(f, sa, sb, acc, std::make_integer_sequence<int, TN * TM>{});
            }
            q = nxt;
        }
    }

    // the wave's partial tile into its own part of the LDS, then every thread adds the waves' partials of
    // its elements in wave order
    f32x4_t* const mine = reinterpret_cast<f32x4_t*>(ring) + lane;
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) mine[(b * TN + a) * 64] = acc[a][b];
    __syncthreads();
    for (int e = threadIdx.x; e < TN * TM * 64; e += 64 * W) {
        f32x4_t v = reinterpret_cast<const f32x4_t*>(smem)[e];
#pragma unroll
        for (int w = 1; w < W; ++w) v += reinterpret_cast<const f32x4_t*>(smem + w * G::WAVE_BYTES)[e];
        const int l = e & 63, t = e >> 6;
        const int m = M0 + 16 * (t / TN) + (l & 15), n = N0 + 16 * (t % TN) + 4 * (l >> 4);
        if (m >= P.M || n >= P.N) continue;
        if constexpr (TOK) v *= P.tok_scale[m];
        *reinterpret_cast<u32x2_t*>(P.Out + (int64_t)m * P.N + n) = (u32x2_t){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
}

template <bool TOK>
void launch_tok(int shape, dim3 grid, hipStream_t st, const Params& P)
{
#define FP8KV_SLICE(I, TN, TM, W, D)                                                                              \
    case I:                                                                                                       \
        static_assert(kSliceShapes[I].tn == TN && kSliceShapes[I].tm == TM && kSliceShapes[I].waves == W, "table"); \
        launch_kernel(gemm_slice_kernel<TN, TM, W, D, TOK>, grid, dim3(64 * W), (SliceGeom<TN, TM, W, D>::LDS), st, P); \
        break
    switch (shape) {
        FP8KV_SLICE(0, 1, 1, 8, 4);
        FP8KV_SLICE(1, 1, 2, 8, 4);
        FP8KV_SLICE(2, 2, 1, 8, 4);
        FP8KV_SLICE(3, 2, 2, 8, 3);
        FP8KV_SLICE(4, 2, 3, 8, 2);
        FP8KV_SLICE(5, 2, 4, 8, 2);
        FP8KV_SLICE(6, 4, 3, 8, 2);
        FP8KV_SLICE(7, 4, 4, 4, 2);
        FP8KV_SLICE(8, 4, 8, 4, 2);
        FP8KV_SLICE(9, 8, 4, 4, 2);
    }
#undef FP8KV_SLICE
}

void launch_slice(int shape, bool tok, dim3 grid, hipStream_t st, const Params& P)
{
    if (tok) launch_tok<true>(shape, grid, st, P);
    else launch_tok<false>(shape, grid, st, P);
}

}  // namespace w4a8_detail
}  // namespace fp8kv
