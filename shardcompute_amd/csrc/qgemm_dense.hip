// Prefill GEMM for many rows: the weights are dequantized once into a bf16 workspace,
// then a dense bf16 MFMA GEMM reads them.
//
//     y[m, n] = sum_k x[m, k] * bf16(s[n, k/64] * q[n, k] + b[n, k/64])
//
// the contraction and the weight rounding of qgemm.hip, whose workgroups each
// dequantize their own weight tile again for every 256 rows of x.
//
// What bounds it: the matrix cores at the clock the power limit leaves (1.5-1.8 GHz
// under this load).  qgemm.hip issues about 100 VALU instructions of dequantization
// per wave and 64-k stage besides its 32 MFMAs and stages x through registers; here
// the stage loop holds MFMAs, LDS reads and LDS-DMA only.  The dequantization costs
// N K (2 + bits/8) bytes of traffic once, which pays from 1000-2000 rows (the rule at
// qgemm_dense_workspace_bytes).  Measured with the dequantization (medians on one box,
// qgemm.hip -> here, W4): 2048 x 28672 x 4096 480 -> 413 us (1166 TFLOP/s), 2048 x 4096 x
// 14336 247 -> 222, 2048 x 6144 x 4096 109 -> 88 (1169), ragged 3821 x 15904 x 8384 964 -> 801
// (1272), 8192 x 7168 x 8192 902 -> 678 (1419); W8 8192 x 7168 x 8192 957 -> 685 (1404).
//
// qgemm_dense_kernel:
// * Workgroup tile 256 x 256 on 4 waves (one per SIMD, each 128 x 128, its 256
//   accumulators in AGPRs) or 256 x 128 on 8 waves (64 x 64 each), for the shapes
//   whose wide tiles would leave the chip idle.  128 x 128 wave tiles read 128 KB of
//   LDS per stage against 192 KB for eight 128 x 64 ones (8192^3: 1473 against 1370
//   TFLOP/s).
// * v_mfma_f32_16x16x32_bf16: half the accumulator traffic of 32x32x16 per flop, and
//   the chip holds a higher clock on it (1.72 against 1.64 GHz, 3-5 % faster).  The
//   weight is operand A, x operand B, so that a lane holds 8 consecutive columns of
//   one row: 16-byte stores (2-byte stores of a column cost 2-4 % at K = 4096).
// * K advances 64 per stage.  Both operands reach LDS by buffer LDS-DMA, two stages,
//   16-byte chunks XOR-swizzled by row.  The operands of a k-step of 32 are read
//   during the step before it; stage g + 2 is issued into the buffer of stage g right
//   after the one barrier of a stage, which follows the last operand read of stage g.
//   Every MFMA slot holds at most one LDS read or one DMA (its M0 write goes before the
//   MFMA): two of them in a slot outlast the 16 cycles of the MFMA (2-3 %).
// * A 4- or 5-stage ring of 32-k stages (more bytes in flight, a barrier per 32) was
//   5 % slower, 32x32x16 MFMAs 3-5 %, DMA spread over both k-steps 8 %.
// * Tiles are dealt to the XCDs in contiguous runs, in column order inside groups of 4 or 8
//   row tiles, so that the 32 tiles an XCD works on share 4 x tiles and 8 weight tiles
//   (or 8 and 4) in its L2.
#include "sc_common.h"
#include "dma_util.h"
#include "gemm_store.h"

#include <type_traits>
#include <utility>

#include "../../include/shardcompute_hip.h"

namespace sc {

namespace {

constexpr int BK = 64;                    // k per stage: one 128-byte row of LDS
constexpr int ROW_BYTES = BK * 2;
constexpr int XCDS = 8;
constexpr int BM = 256;
// columns of weights dequantized at a time: the workspace holds at most this many bytes
constexpr int64_t WS_MAX_BYTES = 256ll << 20;

struct DenseArgs {
    const uint16_t *x;
    const uint16_t *w;        // [N, K] bf16
    const uint16_t *bias;     // null, or by product column
    uint16_t *y;
    int M, N, K;
    int64_t ldy;              // y's row stride
    int n_base;               // column of y (SwiGLU: of the product) that column 0 of w stands for
    int swiglu_i;             // I > 0: columns 2j, 2j + 1 are gate j and up j; y receives act [M, I]
    int mt, nt, tiles;
    int group_m;              // row tiles a run of tiles walks before the next column
};

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// 16-byte chunk c of tile row r sits at position c ^ swz(r) of the row.  An operand read
// covers 16 rows at one chunk per 16 lanes; rows of one parity share 128 bytes of banks
// and have to differ in their 8 positions: 16 consecutive rows of the x tile, rows 8 a + b
// (a, b < 4) of the weight tile.
__device__ __forceinline__ int swz_x(int r) { return (r & 7) ^ ((r >> 3) & 1); }
__device__ __forceinline__ int swz_w(int r) { return ((r >> 1) & 1) | (((r >> 3) & 3) << 1); }

// raw buffer resource: reads past `bytes` return 0
__device__ __forceinline__ u32x4_t buffer_of(const void *p, uint32_t bytes) {
    const uint64_t b = (uint64_t)p;
    u32x4_t r;
    r.x = __builtin_amdgcn_readfirstlane((uint32_t)b);
    r.y = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    r.z = __builtin_amdgcn_readfirstlane(bytes);
    r.w = 0x00020000u;
    return r;
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 16 bytes per lane from buffer + soff + voff to LDS at M0 + 16 * lane.  M0 is written by
// set_m0 at least one instruction earlier (the DMA needs one wait state after it); the
// kernel has no other M0 user.
template <int IMM>
__device__ __forceinline__ void set_m0(uint32_t base) {
    asm volatile("s_add_u32 m0, %0, %1" : : "s"(base), "n"(IMM) : "m0", "scc");
}
__device__ __forceinline__ void dma_lds(u32x4_t buf, uint32_t soff, uint32_t voff) {
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" : : "v"(voff), "s"(buf), "s"(soff) : "memory");
}
#pragma clang diagnostic pop

// D = A B + D with D in AGPRs: with the builtin the register allocator moves a 256-register
// accumulator between AGPRs and VGPRs inside the loop (344 moves a stage).  The compiler
// does not track this MFMA's latency: the s_nop at the end of the stage loop separates it
// from the epilogue's reads.  Its A and B come from LDS reads only, which the compiler
// waits for.
__device__ __forceinline__ void mfma_acc(f32x4_t &c, bf16x8_t a, bf16x8_t b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

template <int I>
using int_c = std::integral_constant<int, I>;
template <class F, int... Is>
__device__ __forceinline__ void for_each_slot(F &&f, std::integer_sequence<int, Is...>) {
    (f(int_c<Is>{}), ...);
}

}  // namespace

template <int BN, int WGM, int WGN>
__global__ void __launch_bounds__(64 * WGM * WGN) __attribute__((amdgpu_waves_per_eu(WGM * WGN / 4, WGM * WGN / 4)))
qgemm_dense_kernel(DenseArgs a) {
    constexpr int WAVES = WGM * WGN;
    constexpr int WM = BM / WGM, WN = BN / WGN;          // wave tile
    constexpr int NI = WM / 16, NJ = WN / 16;
    constexpr int NM = NI * NJ;                          // MFMAs per 32-k step
    constexpr int NR = NI + NJ;                          // operand reads per step
    constexpr int STAGE = (BM + BN) * ROW_BYTES;
    constexpr int AI = BM / 8 / WAVES, BI = BN / 8 / WAVES, ND = AI + BI;   // DMA instructions per wave and stage
    constexpr int SD = NM / ND;                          // DMA d sits in slot SD d + (SD / 2 | 1) of step 1
    constexpr int SR = NM / 2 / NR > 0 ? NM / 2 / NR : 1;
    static_assert((ND - 1) * SD + (SD / 2 | 1) < NM, "every DMA of a stage has its slot");
    static_assert((NR - 1) * SR < NM, "every operand read of a step has its slot");
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lq = lane >> 4;
    const int wm = w / WGN, wn = w % WGN;
    const int M = a.M, N = a.N, K = a.K;

    // workgroup i runs on XCD i % 8: that XCD takes the tiles [x per, (x + 1) per)
    const int per = (int)(gridDim.x / XCDS);
    const int tile = (int)(blockIdx.x % XCDS) * per + (int)(blockIdx.x / XCDS);
    if (tile >= a.tiles) return;
    const int grp = tile / (a.group_m * a.nt), first = grp * a.group_m;
    const int rows = min(a.group_m, a.mt - first), in = tile - grp * a.group_m * a.nt;
    const int m0 = (first + in % rows) * BM, n0 = in / rows * BN;

    // DMA instruction i of this wave covers 8 tile rows; lane l lands at row l / 8,
    // position l % 8, and loads the chunk the swizzle puts there (rows past the matrix
    // load its last row; they are never stored)
    uint32_t va[AI], vb[BI];
#pragma unroll
    for (int i = 0; i < AI; ++i) {
        const int r = (w * AI + i) * 8 + (lane >> 3), c = (lane & 7) ^ swz_x(r);
        va[i] = (uint32_t)min(r, M - 1 - m0) * (uint32_t)(K * 2) + c * 16;
    }
#pragma unroll
    for (int i = 0; i < BI; ++i) {
        const int r = (w * BI + i) * 8 + (lane >> 3), c = (lane & 7) ^ swz_w(r);
        vb[i] = (uint32_t)min(r, N - 1 - n0) * (uint32_t)(K * 2) + c * 16;
    }
    const u32x4_t xbuf = buffer_of(a.x + (size_t)m0 * K, (uint32_t)min(BM, M - m0) * (uint32_t)(K * 2));
    const u32x4_t wbuf = buffer_of(a.w + (size_t)n0 * K, (uint32_t)min(BN, N - n0) * (uint32_t)(K * 2));
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const uint32_t lds_a = __builtin_amdgcn_readfirstlane(lds0 + w * (AI * 1024));
    const uint32_t lds_b = __builtin_amdgcn_readfirstlane(lds0 + BM * ROW_BYTES + w * (BI * 1024));

    f32x4_t acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{};
    bf16x8_t af[2][NI], bf[2][NJ];
    // Operand reads, k chunk 4 ks + lq.  x: rows 16 i + li of the wave's tile.  Weights:
    // block j's row li is row 32 (j / 2) + 8 (li / 4) + 4 (j % 2) + li % 4, so that the
    // accumulators of blocks 2 p and 2 p + 1 of a lane are 8 consecutive columns.
    uint32_t ra[2], rb[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const int rx = wm * WM + li;
        ra[ks] = rx * ROW_BYTES + (((ks * 4 + lq) ^ swz_x(rx)) << 4);
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            const int rw = wn * WN + 8 * (li >> 2) + 4 * o + (li & 3);
            rb[ks][o] = (BM + rw) * ROW_BYTES + (((ks * 4 + lq) ^ swz_w(rw)) << 4);
        }
    }
    auto read = [&](int buf, int ks, int p, int i) __attribute__((always_inline)) {
        const uint8_t *s = smem + buf * STAGE;
        if (i < NJ) bf[p][i] = as_bf16x8(*reinterpret_cast<const uint4 *>(s + rb[ks][i & 1] + (i >> 1) * (32 * ROW_BYTES)));
        else af[p][i - NJ] = as_bf16x8(*reinterpret_cast<const uint4 *>(s + ra[ks] + (i - NJ) * (16 * ROW_BYTES)));
    };

    const int G = K / BK, gl = G - 1;
    // stages 0 and 1
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        const uint32_t so = (uint32_t)min(st, gl) * ROW_BYTES;
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const uint32_t l = (i < AI ? lds_a + i * 1024 : lds_b + (i - AI) * 1024) + st * STAGE;
            set_m0<0>(l);
            asm volatile("s_nop 0");
            if (i < AI) dma_lds(xbuf, so, va[i < AI ? i : 0]);
            else dma_lds(wbuf, so, vb[i >= AI ? i - AI : 0]);
        }
    }
    dma::wait_vm<ND>();
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int i = 0; i < NR; ++i) read(0, 0, 0, i);

    // step KS of stage g (buffer buf): its MFMAs, the reads of the next step's operands
    // and, in step 1, the DMA of stage g + 2 into this stage's buffer.  Past the last
    // stage the DMA repeats that stage into the buffer nobody reads and the reads
    // fetch operands nobody uses, so the loop has no branches.
    auto step = [&](int g, int buf, auto ks_tag) __attribute__((always_inline)) {
        constexpr int ks = decltype(ks_tag)::value;
        if (ks == 1) {
            // this wave's part of stage g + 1 has landed and its last operands of stage g
            // are in registers; after the barrier both hold for every wave
            dma::wait_vm<0>();
            dma::wait_lgkm0();
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
        const uint32_t so = (uint32_t)min(g + 2, gl) * ROW_BYTES;
        const uint32_t la = lds_a + buf * STAGE, lb = lds_b + buf * STAGE;
        auto slot = [&](auto i_tag) __attribute__((always_inline)) {
            constexpr int i = decltype(i_tag)::value;
            constexpr int d = i / SD;
            constexpr bool D = ks == 1 && i % SD == (SD / 2 | 1) && d < ND;
            if constexpr (D) {
                if constexpr (d < AI) set_m0<d * 1024>(la);
                else set_m0<(d - AI) * 1024>(lb);
            }
            mfma_acc(acc[i / NJ][i % NJ], bf[ks][i % NJ], af[ks][i / NJ]);
            if constexpr (i % SR == 0 && i / SR < NR) {
                if constexpr (ks == 0) read(buf, 1, 1, i / SR);
                else read(buf ^ 1, 0, 0, i / SR);
            }
            if constexpr (D) {
                if constexpr (d < AI) dma_lds(xbuf, so, va[d]);
                else dma_lds(wbuf, so, vb[d - AI]);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        for_each_slot(slot, std::make_integer_sequence<int, NM>{});
    };
    int buf = 0, g = 0;
    do {
        step(g, buf, int_c<0>{});
        step(g, buf, int_c<1>{});
        // the latency of the last MFMA before anything can read its result (11 wait
        // states for 16x16x32), inside the loop because the compiler, which does not see
        // it, may move accumulators right behind the loop; in the loop it hides behind the
        // MFMA's own 16 cycles
        asm volatile("s_nop 10");
        buf ^= 1;
    } while (++g < G);
    dma::wait_vm<0>();       // no DMA may land after the workgroup has ended

    // ---- epilogue: acc[i][2 p] and acc[i][2 p + 1] of lane (li, lq) are row
    // m0 + wm WM + 16 i + li, columns n0 + wn WN + 32 p + 8 lq .. + 7, rounded to bf16, the
    // bias added and rounded again
    // INNER: a tile inside the matrix, no bias (predicates for all cost 0.5 % of a product)
    auto store = [&](auto inner_tag, auto swiglu_tag) __attribute__((always_inline)) {
        constexpr bool INNER = decltype(inner_tag)::value != 0, SWIGLU = decltype(swiglu_tag)::value != 0;
        const int nl = n0 + wn * WN + 8 * lq;
        uint32_t bb[NJ / 2][4] = {};
        if (!INNER && a.bias) {
#pragma unroll
            for (int p = 0; p < NJ / 2; ++p)
                load_bias8<SWIGLU>(bb[p], a.bias, a.n_base + nl + 32 * p, nl + 32 * p, N, a.swiglu_i);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int m = m0 + wm * WM + 16 * i + li;
            if (!INNER && m >= M) continue;
            uint16_t *yr = a.y + (size_t)m * a.ldy;
#pragma unroll
            for (int p = 0; p < NJ / 2; ++p) {
                uint32_t o[4] = {cvt_pk_bf16(acc[i][2 * p][0], acc[i][2 * p][1]),
                                 cvt_pk_bf16(acc[i][2 * p][2], acc[i][2 * p][3]),
                                 cvt_pk_bf16(acc[i][2 * p + 1][0], acc[i][2 * p + 1][1]),
                                 cvt_pk_bf16(acc[i][2 * p + 1][2], acc[i][2 * p + 1][3])};
                store_cols8<INNER, SWIGLU>(o, yr, a.n_base + nl + 32 * p, nl + 32 * p, N, a.bias != nullptr, bb[p]);
            }
        }
    };
    const bool inner = !a.bias && m0 + BM <= M && n0 + BN <= N;
    if (a.swiglu_i) {
        if (inner) store(int_c<1>{}, int_c<1>{});
        else store(int_c<0>{}, int_c<1>{});
    } else {
        if (inner) store(int_c<1>{}, int_c<0>{});
        else store(int_c<0>{}, int_c<0>{});
    }
}

// Rows [r0, r0 + rows) of the product's weights as bf16 [rows, K].  half = I > 0: product
// row 2j is weight row j (gate), 2j + 1 row I + j (up).  A wave takes one row, 8 codes and
// a 16-byte store per lane and iteration, so loads and stores are contiguous; bound by the
// stores (24576 x 4096 W4: 46 us, 5.4 TB/s read and written).
template <int BITS>
__global__ void __launch_bounds__(256) dequant_rows_kernel(const uint32_t *wq, const uint16_t *s, const uint16_t *b,
                                                           int K, int r0, int rows, int half, uint16_t *out) {
    const int lane = threadIdx.x & 63;
    const int r = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6);
    if (r >= rows) return;
    const int pr = r0 + r;
    const int row = half ? (pr >> 1) + (pr & 1) * half : pr;
    const uint32_t *src = wq + (size_t)row * ((size_t)K * BITS / 32);
    const uint16_t *sr = s + (size_t)row * (K / 64), *br = b + (size_t)row * (K / 64);
    uint16_t *dst = out + (size_t)r * K;
    const int U = K / 8;                    // units of 8 codes
    uint32_t nib = 0x0F0F0F0Fu;             // opaque: one v_cvt_f32_ubyteN per code
    asm volatile("" : "+s"(nib));
#pragma unroll 4
    for (int u = lane; u < U; u += 64) {
        const float sf = bf2f(sr[u >> 3]), bf = bf2f(br[u >> 3]);
        uint32_t o[4];
        if (BITS == 4) {
            const uint32_t v = src[u], lo = v & nib, hi = (v >> 4) & nib;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[j] = cvt_pk_bf16(fmaf(sf, ubyte_f32(lo, j), bf), fmaf(sf, ubyte_f32(hi, j), bf));
        } else {
            const uint2 v = *reinterpret_cast<const uint2 *>(src + 2 * u);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t c = j < 2 ? v.x : v.y;
                o[j] = cvt_pk_bf16(fmaf(sf, ubyte_f32(c, 2 * (j & 1)), bf), fmaf(sf, ubyte_f32(c, 2 * (j & 1) + 1), bf));
            }
        }
        *reinterpret_cast<uint4 *>(dst + 8 * u) = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

template <int BN, int WGM, int WGN>
static int launch_dense_cols(const DenseArgs &full, int n0, int nc, hipStream_t stream) {
    DenseArgs a = full;
    a.w = full.w + (size_t)n0 * full.K;
    a.n_base = full.n_base + n0;
    a.N = nc;
    a.nt = (nc + BN - 1) / BN;
    const int64_t tiles = (int64_t)a.mt * a.nt;
    if (tiles > 0x7FFFFFF0) return set_error(SC_EINVAL, "qgemm_dense: grid too large");
    a.tiles = (int)tiles;
    // 8 row tiles where the launch is one round, 4 otherwise (measured, 4 -> 8: 2048 x 4096 x
    // 4096 73.4 -> 70.3 us, x 6144 94.2 -> 91.4, but 2048 x 28672 x 4096 440 -> 444; 2 is
    // slower everywhere, 8192 x 7168 x 8192 689 -> 739)
    a.group_m = tiles <= device_info().num_cus ? 8 : 4;
    constexpr int LDS = 2 * (BM + BN) * ROW_BYTES;
    auto kern = qgemm_dense_kernel<BN, WGM, WGN>;
    static bool configured = false;
    if (!configured) {
        SC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        configured = true;
    }
    const unsigned blocks = (unsigned)((tiles + XCDS - 1) / XCDS * XCDS);
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * WGM * WGN), LDS, stream, a);
    SC_HIP_CHECK(hipGetLastError());
    return SC_OK;
}

// The columns [0, wide) of a launch of mt row tiles run as 256 x 256 tiles, the others as
// 256 x 128 ones; cost: the estimate in hundredths of a round of wide tiles.
struct DensePlan {
    int wide;
    int64_t cost;
};

// Wide tiles, narrow ones, or whole rounds of wide ones and the last columns narrow: the
// shortest estimate of rounds x tile time, a 256 x 128 tile taking 0.7 of a 256 x 256 one (one
// round at M = 2048, K 2048, 4096, 8192: narrow 37, 68, 122 us, wide 53, 94, 176).  Measured
// against the rule before, 0.64 and a mixed launch only where the last round splits evenly
// (W4): 1.5 rounds, mixed, 3031 x 7680 x 3968 185 -> 162 us; 2 wide rounds where 3 narrow
// ones ran, 1680 x 13760 x 7808 453 -> 371.
static DensePlan plan_dense(int mt, int64_t cols) {
    const int cus = device_info().num_cus;
    const auto rounds = [&](int64_t n, int bn) { return ((int64_t)mt * ((n + bn - 1) / bn) + cus - 1) / cus; };
    DensePlan best{(int)cols, 100 * rounds(cols, 256)};
    const int64_t full = (int64_t)mt * ((cols + 255) / 256) / cus;      // whole rounds of wide tiles,
    const int64_t n1 = full * cus / mt * 256;                           // the columns they hold
    for (const int64_t w : {(int64_t)0, n1}) {
        if (w >= cols) continue;
        const int64_t cost = (w ? 100 * full : 0) + 70 * rounds(cols - w, 128);
        if (cost < best.cost) best = DensePlan{(int)w, cost};
    }
    return best;
}

static int launch_dense(const DenseArgs &a, hipStream_t stream) {
    const int w = plan_dense(a.mt, a.N).wide;
    if (w > 0) {
        const int rc = launch_dense_cols<256, 2, 2>(a, 0, w, stream);
        if (rc || w == a.N) return rc;
    }
    return launch_dense_cols<128, 4, 2>(a, w, a.N - w, stream);
}

// Bytes of workspace the dense path wants for a product, 0 where the fused GEMM is the
// faster (or the shape is not taken).  The dequantization's cost is per weight and two
// launches, the gain per product element, and a dense tile is slower to start and end, so
// the line is drawn at 2^23 outputs (128 wide tiles, half the CUs), 1280 rows; from 1024
// rows at 11.5 M outputs, K up to 8192 (above, the dequantization is a sixth of the time and
// the two tie: 1057 x 12544 x 11072 340 -> 348, 1143 x 18672 x 10752 537 -> 525); and with K
// below 2048, where start and end weigh more, 20 M, below 1536 26 M.
// Measured at the line, fused GEMM -> here, W4 (W8), us: 2048 x 4096 x 4096 77 -> 72
// (78 -> 71), 1536 x 4096 x 4096 65 -> 67, 1280 x 8192 x 3584 96 -> 86, 1024 x 8192 x 3584
// 70 -> 70 (69 -> 71), 1024 x 11264 x 2048 63 -> 62 (65 -> 58), 4096 x 2048 x 5632
// 103 -> 93, 3072 x 2048 x 5632 90 -> 89, 3178 x 8448 x 1024 71 -> 65, 6144 x 4096 x 1024
// 60 -> 62, 1024 x 22528 x 1280 69 -> 71, 4096 x 2560 x 2048 56 -> 51, 3072 x 2560 x 2048
// 40 -> 43.  Over 900 sizes above the line 1.21 times as fast on the average, one of them
// slower by over 2 % (3 %).
int64_t qgemm_dense_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M < 1024 || M > (1 << 30) || N < 256 || N > (1 << 30) || K < 1024 || K > (1 << 20) || K % BK || N % 8) return 0;
    if (M < 1280 && K > 8192) return 0;
    if (M * N < (K < 1536 ? 26000000 : K < 2048 ? 20000000 : M < 1280 ? 11500000 : 1 << 23)) return 0;
    const int64_t row = K * 2;
    int64_t rows = N;
    if (rows * row > WS_MAX_BYTES) rows = WS_MAX_BYTES / row / 256 * 256;   // whole 256-column tiles at a time
    return rows < 256 ? 0 : rows * row;
}

// SC_EUNSUPPORTED (nothing launched): the shape, or a workspace that is missing, too small or misaligned
int launch_qgemm_dense(const uint16_t *x, const uint32_t *wq, const uint16_t *s, const uint16_t *b,
                       const uint16_t *bias, uint16_t *y, int M, int N, int K, int bits, hipStream_t stream,
                       int swiglu_half, void *ws, int64_t ws_bytes) {
    const int64_t need = qgemm_dense_workspace_bytes(M, N, K);
    if (need == 0 || !ws || ws_bytes < need || ((uintptr_t)ws % 16) != 0) return SC_EUNSUPPORTED;
    if ((bits != 4 && bits != 8) || (swiglu_half && N != 2 * swiglu_half)) return SC_EUNSUPPORTED;
    if (!wide_rows(y, N, swiglu_half)) return SC_EUNSUPPORTED;
    if (device_info().max_lds_per_block < 2 * (BM + 256) * ROW_BYTES) return SC_EUNSUPPORTED;
    int rows = (int)(need / ((int64_t)K * 2));
    DenseArgs a;
    a.x = x; a.w = static_cast<const uint16_t *>(ws); a.bias = bias; a.y = y;
    a.M = M; a.K = K;
    a.ldy = swiglu_half ? swiglu_half : N;
    a.swiglu_i = swiglu_half;
    a.mt = (M + BM - 1) / BM;
    a.nt = a.tiles = 0;
    if (rows < N) {
        // Several chunks of columns: whole rounds of wide tiles each (W4 1854 x 13120 x 11456,
        // 620 us on the fused GEMM, two chunks of the largest size 796, so 546).  Where the
        // chunks' rounds still come to much more than the whole product's, the fused GEMM
        // (1033 x 25280 x 11200, three chunks of 0.9, 0.9 and 0.7 rounds for 2: 663 -> 801).
        const int64_t cus = device_info().num_cus, full = a.mt * (rows / 256) / cus;
        if (full * cus / a.mt > 0) rows = (int)(full * cus / a.mt * 256);
        int64_t cost = 0;
        for (int n0 = 0; n0 < N; n0 += rows) cost += plan_dense(a.mt, N - n0 < rows ? N - n0 : rows).cost;
        if (100 * cost > 115 * plan_dense(a.mt, N).cost) return SC_EUNSUPPORTED;
    }
    for (int n0 = 0; n0 < N; n0 += rows) {
        const int nc = N - n0 < rows ? N - n0 : rows;
        const dim3 grid((unsigned)((nc + 3) / 4)), block(256);
        if (bits == 4)
            hipLaunchKernelGGL(dequant_rows_kernel<4>, grid, block, 0, stream, wq, s, b, K, n0, nc, swiglu_half,
                               static_cast<uint16_t *>(ws));
        else
            hipLaunchKernelGGL(dequant_rows_kernel<8>, grid, block, 0, stream, wq, s, b, K, n0, nc, swiglu_half,
                               static_cast<uint16_t *>(ws));
        SC_HIP_CHECK(hipGetLastError());
        a.N = nc;
        a.n_base = n0;
        const int rc = launch_dense(a, stream);
        if (rc) return rc;
    }
    return SC_OK;
}

}  // namespace sc
