// GEMM of a few hundred rows on 128 x 128 tiles.
//
//     y[m, n] = sum_k x[m, k] * bf16(s[n, k/64] * q[n, k] + b[n, k/64])
//
// the contraction and the weight rounding of qgemm.hip, for the products whose 256-row tiles
// leave CUs idle or rows empty and are too small for qgemm_dense.hip.
//
// What bounds it: a stage's chain (barrier, LDS reads, dequantization, MFMAs: 0.75 us, of
// which the MFMAs 0.25) with one wave per SIMD; its gain is the smaller tile, a 256-row
// tile's stage takes 0.95-1.1 us there and leaves rows empty.
//
// * A workgroup is 4 waves and 128 x 128 outputs.  Wave w owns the 32 weight rows
//   [32 w, 32 w + 32) and all 128 rows of x, on v_mfma_f32_16x16x32_bf16 with the
//   weights as operand A: each weight is dequantized once per workgroup, straight into the
//   operand, and only x and the packed codes pass through LDS.
// * K advances 64 per stage, everything by LDS-DMA two stages ahead into 3-slot rings (x
//   rows of 128 bytes, 16-byte chunks XOR-swizzled; the wave's own code rows; every 8
//   stages the wave's scales and biases of 8 groups): one vmcnt wait and one barrier a stage.
//   (The list before a block's has one instruction more; waiting as if it had not is safe.)
// * Lane part lq's k-step ks takes k chunk 2 lq + ks of the stage, for x and codes alike, so
//   that a lane's codes of a stage are 8 (W4) or 16 (W8) consecutive bytes.
// * Weight block j's row li is row 8 (li / 4) + 4 j + li % 4 of the wave's 32, so that a lane
//   ends with 8 consecutive columns of a row: 16-byte stores.
// * Few tiles split K over the grid's second dimension (fp32 partials, split-K pass).
// * Every operand read of a stage goes out before its DMA issue and arithmetic (read by read
//   before each MFMA: 29 instead of 27 us), and the stages are one rolled loop (unrolled by 8
//   for the scales it spilled, and each spill reload waited for the DMA too: 41 us).
// Measured (2048 -> 2560 W4): 170 rows 31.8 -> 26.3 us, 768 rows 31.5 -> 27.2; 5632 -> 2048, 333
// rows 33.8 -> 27.7.
#include "sc_common.h"
#include "dma_util.h"
#include "gemm_store.h"
#include "../../include/shardcompute_hip.h"

#include <type_traits>

namespace sc {

namespace {

constexpr int MB = 128, NB = 128;          // tile
constexpr int XCDS = 8, GROUP_M = 8;
constexpr int NX = 3;                      // ring slots: stage g being read, g + 1 and g + 2 landing
constexpr int XT = MB * 128;               // x stage: 16 KB

template <int BITS>
struct MidGeo {
    static constexpr int CR = 64 * BITS / 8;               // code bytes of a row and stage (32 or 64)
    static constexpr int CT = NB * CR;                     // codes of a stage: 4 or 8 KB
    static constexpr int CI = CT / 1024 / 4;               // code DMA instructions per wave and stage
    static constexpr int XI = XT / 1024 / 4;               // x DMA instructions per wave and stage
    static constexpr int LI = CI + XI;                     // a stage's list (one more where a block starts)
    static constexpr int O_C = NX * XT, O_SB = O_C + NX * CT;
    static constexpr int LDS = O_SB + 2 * 4096;            // two blocks of 128 rows' scales and biases
};

struct MidArgs {
    const uint16_t *x;
    const uint8_t *wq;
    const uint16_t *s, *b;
    const uint16_t *bias;
    uint16_t *y;
    float *partials;          // [splits, M, N] fp32, or null: y is written directly
    int M, N, K, G;
    int gps;                  // groups per K split, a multiple of 8
    int64_t ldy;
    int swiglu_i;             // I > 0: product columns 2j, 2j + 1 are weight rows j and I + j
    int mt, nt, tiles;
};

__device__ __forceinline__ int mid_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

}  // namespace

template <int BITS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) qgemm_mid_kernel(MidArgs a) {
    using C = MidGeo<BITS>;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lq = lane >> 4;
    const int M = a.M, N = a.N, K = a.K;

    // workgroup i runs on XCD i % 8: that XCD takes a contiguous run of tiles, in column
    // order inside groups of GROUP_M row tiles
    const int per = (int)(gridDim.x / XCDS);
    const int tile = (int)(blockIdx.x % XCDS) * per + (int)(blockIdx.x / XCDS);
    if (tile >= a.tiles) return;
    const int grp = tile / (GROUP_M * a.nt), first = grp * GROUP_M;
    const int rows = min(GROUP_M, a.mt - first), in = tile - grp * GROUP_M * a.nt;
    const int m0 = (first + in % rows) * MB, n0 = in / rows * NB;
    const int g0 = (int)blockIdx.y * a.gps, ng = min(a.G - g0, a.gps);

    // weight row of product column c (columns past the matrix repeat its last)
    auto wrow = [&](int c) {
        c = min(c, N - 1);
        return a.swiglu_i ? (c >> 1) + (c & 1) * a.swiglu_i : c;
    };
    // DMA sources of this lane; lane l of an instruction lands 16 l bytes after its base
    const uint8_t *xsrc = reinterpret_cast<const uint8_t *>(a.x) + ((size_t)m0 * K + (size_t)g0 * 64) * 2;
    uint32_t xoff[C::XI];
#pragma unroll
    for (int i = 0; i < C::XI; ++i) {
        const int r = 32 * w + 8 * i + (lane >> 3), c = (lane & 7) ^ mid_swz(r);
        xoff[i] = (uint32_t)min(r, M - 1 - m0) * (uint32_t)(K * 2) + 16 * c;
    }
    constexpr int CPR = C::CR / 16, RPI = 64 / CPR;        // 16-byte pieces of a code row, rows an instruction
    const uint8_t *csrc[C::CI];
#pragma unroll
    for (int i = 0; i < C::CI; ++i)
        csrc[i] = a.wq + (size_t)wrow(n0 + 32 * w + RPI * i + lane / CPR) * ((size_t)K * BITS / 8) +
                  (size_t)g0 * C::CR + 16 * (lane % CPR);
    const uint8_t *sbsrc = reinterpret_cast<const uint8_t *>(lane < 32 ? a.s : a.b) +
                           ((size_t)wrow(n0 + 32 * w + (lane & 31)) * a.G + g0) * 2;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const uint32_t lx = lds0 + w * (C::XI * 1024), lc = lds0 + C::O_C + w * (C::CI * 1024), lsb = lds0 + C::O_SB + w * 1024;
    // list t: the scales and biases of block t / 8 where it starts, the codes and x of stage t
    // (stages past the split repeat the last one into slots nobody reads any more)
    auto issue = [&](int t, int slot, bool sb) __attribute__((always_inline)) {
        const int tc = min(t, ng - 1);
        if (sb) dma::dma16(sbsrc + 16 * min(t >> 3, (ng >> 3) - 1), lsb + ((t >> 3) & 1) * 4096);
#pragma unroll
        for (int i = 0; i < C::CI; ++i) dma::dma16(csrc[i] + (size_t)tc * C::CR, lc + slot * C::CT + i * 1024);
#pragma unroll
        for (int i = 0; i < C::XI; ++i)
            dma::dma16s(xsrc + (size_t)tc * 128, xoff[i], lx + slot * XT + i * 1024);
    };

    f32x4_t acc[8][2];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4_t{};
    uint32_t nib = 0x0F0F0F0Fu;                            // opaque: one v_cvt_f32_ubyteN per code
    asm volatile("" : "+s"(nib));
    int wr[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) wr[j] = 8 * (li >> 2) + 4 * j + (li & 3);
    uint32_t xo[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) xo[ks] = (uint32_t)(li * 128 + (((2 * lq + ks) ^ mid_swz(li)) << 4));

    issue(0, 0, true);
    issue(1, 1, false);
    int slot = 0;
#pragma clang loop unroll(disable)
    for (int g = 0; g < ng; ++g) {
        // list g has landed (list g + 1 is in flight); after the barrier every wave's part
        // has, and stage g - 1's slot is free for list g + 2
        dma::wait_vm<C::LI>();
        __syncthreads();
        const uint8_t *sb = smem + C::O_SB + ((g >> 3) & 1) * 4096 + w * 1024 + 2 * (g & 7);
        float sf[2], bf[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            sf[j] = bf2f(*reinterpret_cast<const uint16_t *>(sb + 16 * wr[j]));
            bf[j] = bf2f(*reinterpret_cast<const uint16_t *>(sb + 512 + 16 * wr[j]));
        }
        const uint8_t *xs = smem + slot * XT;
        const uint8_t *cs = smem + C::O_C + slot * C::CT + w * (C::CI * 1024);
        uint32_t cw[2][BITS == 4 ? 2 : 4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (BITS == 4) {
                const uint2 v = *reinterpret_cast<const uint2 *>(cs + wr[j] * 32 + 8 * lq);
                cw[j][0] = v.x; cw[j][1] = v.y;
            } else {
                const uint4 v = *reinterpret_cast<const uint4 *>(cs + wr[j] * 64 + 16 * lq);
                cw[j][0] = v.x; cw[j][1] = v.y; cw[j][2] = v.z; cw[j][3] = v.w;
            }
        }
        // every operand read before the DMA issue and the arithmetic, in the order of use: the
        // scheduler otherwise places each read in front of its MFMA and waits it out
        bf16x8_t xf[2][8];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 8; ++i)
                xf[ks][i] = as_bf16x8(*reinterpret_cast<const uint4 *>(xs + xo[ks] + i * (16 * 128)));
        __builtin_amdgcn_sched_barrier(0);
        issue(g + 2, slot == 0 ? 2 : slot - 1, (g & 7) == 6);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            bf16x8_t wf[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                uint32_t o[4];
                if constexpr (BITS == 4) {
                    const uint32_t lo = cw[j][ks] & nib, hi = (cw[j][ks] >> 4) & nib;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        o[e] = cvt_pk_bf16(fmaf(sf[j], ubyte_f32(lo, e), bf[j]), fmaf(sf[j], ubyte_f32(hi, e), bf[j]));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t v = cw[j][2 * ks + (e >> 1)];
                        o[e] = cvt_pk_bf16(fmaf(sf[j], ubyte_f32(v, 2 * (e & 1)), bf[j]),
                                           fmaf(sf[j], ubyte_f32(v, 2 * (e & 1) + 1), bf[j]));
                    }
                }
                wf[j] = as_bf16x8(o[0], o[1], o[2], o[3]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], xf[ks][i], acc[i][j], 0, 0, 0);
        }
        slot = slot == 2 ? 0 : slot + 1;
    }
    dma::wait_vm<0>();                                     // no DMA may land after the workgroup ends

    // ---- acc[i][0], acc[i][1] of lane (li, lq): row m0 + 16 i + li, columns n0 + 32 w + 8 lq .. + 7
    const int n = n0 + 32 * w + 8 * lq;
    if (n >= N) return;
    if (a.partials) {
        float *pz = a.partials + (size_t)blockIdx.y * M * N;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int m = m0 + 16 * i + li;
            if (m >= M) continue;
            float *p = pz + (size_t)m * N + n;
#pragma unroll
            for (int j = 0; j < 2; ++j)
                *reinterpret_cast<float4 *>(p + 4 * j) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
        }
        return;
    }
    auto store = [&](auto swiglu_tag) __attribute__((always_inline)) {
        constexpr bool SWIGLU = decltype(swiglu_tag)::value;
        uint32_t bb[4] = {};
        if (a.bias) load_bias8<SWIGLU>(bb, a.bias, n, n, N, a.swiglu_i);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int m = m0 + 16 * i + li;
            if (m >= M) continue;
            uint32_t o[4] = {cvt_pk_bf16(acc[i][0][0], acc[i][0][1]), cvt_pk_bf16(acc[i][0][2], acc[i][0][3]),
                             cvt_pk_bf16(acc[i][1][0], acc[i][1][1]), cvt_pk_bf16(acc[i][1][2], acc[i][1][3])};
            store_cols8<false, SWIGLU>(o, a.y + (size_t)m * a.ldy, n, n, N, a.bias != nullptr, bb);
        }
    };
    if (a.swiglu_i) store(std::true_type{});
    else store(std::false_type{});
}

template <int BITS>
static int launch_mid_t(const MidArgs &a, int splits, hipStream_t stream) {
    auto kern = qgemm_mid_kernel<BITS>;
    constexpr int LDS = MidGeo<BITS>::LDS;
    static bool configured = false;
    if (!configured) {
        SC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        configured = true;
    }
    const unsigned blocks = (unsigned)((a.tiles + XCDS - 1) / XCDS * XCDS);
    hipLaunchKernelGGL(kern, dim3(blocks, (unsigned)splits), dim3(256), LDS, stream, a);
    SC_HIP_CHECK(hipGetLastError());
    return SC_OK;
}

// K splits of a product of `tiles` tiles, a quarter of the CUs at most, over nb >= 8
// scale/bias blocks: about one workgroup a CU, at least 16 stages each
static int mid_splits(int64_t tiles, int nb) {
    int ks = (int)(device_info().num_cus / tiles);
    if (ks > nb / 2) ks = nb / 2;
    const int bps = (nb + ks - 1) / ks;
    return (nb + bps - 1) / bps;
}

// SC_EUNSUPPORTED (nothing launched) when the shape is not taken.
int launch_qgemm_mid(const uint16_t *x, const uint32_t *wq, const uint16_t *s, const uint16_t *b,
                     const uint16_t *bias, uint16_t *y, int M, int N, int K, int bits, hipStream_t stream,
                     int swiglu_half, bool no_alloc) {
    if (K % 512 || M < 1 || N < 1 || (int64_t)K > (1 << 20)) return SC_EUNSUPPORTED;
    if ((bits != 4 && bits != 8) || (swiglu_half && N != 2 * swiglu_half)) return SC_EUNSUPPORTED;
    if (!wide_rows(y, N, swiglu_half)) return SC_EUNSUPPORTED;
    if (((uintptr_t)x | (uintptr_t)wq | (uintptr_t)s | (uintptr_t)b) % 16) return SC_EUNSUPPORTED;
    if (device_info().max_lds_per_block < MidGeo<8>::LDS) return SC_EUNSUPPORTED;
    MidArgs a;
    a.x = x; a.wq = reinterpret_cast<const uint8_t *>(wq); a.s = s; a.b = b; a.bias = bias; a.y = y;
    a.partials = nullptr;
    a.M = M; a.N = N; a.K = K; a.G = K / 64; a.gps = a.G;
    a.ldy = swiglu_half ? swiglu_half : N;
    a.swiglu_i = swiglu_half;
    a.mt = (M + MB - 1) / MB;
    a.nt = (N + NB - 1) / NB;
    const int64_t tiles = (int64_t)a.mt * a.nt;
    // One workgroup a CU: a stage takes 0.75 us alone and two workgroups of a CU gain little
    // from each other (340 tiles 40 us where 120 take 27).  From K = 4096, where qgemm.hip
    // splits K as well, a quarter of that.  Measured, qgemm.hip -> here, us (W4): K = 2048,
    // 170 x 2560 (40 tiles) 32 -> 26, 768 x 2560 (120) 32 -> 27, 170 x 11264 (176) 32 -> 27,
    // 333 x 11264 (264) 34 -> 37, 2103 x 2560 (340) 36 -> 41; 5632 -> 2048 333 rows (48)
    // 34 -> 28, 768 rows (96) 44 -> 46; 4096 -> 6144 170 rows (96) 34 -> 35.
    if (tiles > (K < 4096 ? device_info().num_cus : device_info().num_cus / 4)) return SC_EUNSUPPORTED;
    a.tiles = (int)tiles;
    // K is split from 4096 on, where qgemm.hip splits each of these products too (its 256-wide
    // tiles are no more than these, a quarter of the CUs), because the partials live in the
    // library's scratch.  No-alloc partials beyond the fixed array: K whole.
    int splits = K >= 4096 ? mid_splits(tiles, a.G / 8) : 1;
    const size_t need = (size_t)splits * M * N;
    if (splits > 1 && no_alloc && need * sizeof(float) > (size_t)SC_QMM_NOALLOC_SCRATCH_BYTES) splits = 1;
    if (splits == 1) return bits == 4 ? launch_mid_t<4>(a, 1, stream) : launch_mid_t<8>(a, 1, stream);
    SplitKScratch ws;
    int rc = no_alloc ? qmm_noalloc_scratch(&ws.partials) : splitk_scratch(need, 1, &ws);
    if (rc) return rc;
    a.partials = ws.partials;
    a.swiglu_i = 0;                                        // natural columns; the pass applies SwiGLU
    a.gps = (a.G / 8 + splits - 1) / splits * 8;
    rc = bits == 4 ? launch_mid_t<4>(a, splits, stream) : launch_mid_t<8>(a, splits, stream);
    if (rc) return rc;
    return launch_qmm_finalize(ws.partials, splits, M, N, bias, y, swiglu_half, stream);
}

}  // namespace sc
