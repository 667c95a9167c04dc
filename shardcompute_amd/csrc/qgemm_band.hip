// Kernel C: the middle band of the quantized product, 8 <= M <= 256 rows of x.
//
// y[m, n] = sum_k x[m, k] * (s[n, k/64] * q[n, k] + b[n, k/64])
// (mx.quantized_matmul(x, wq, s, b, transpose=True, group_size=64, bits),
//  src/shardcompute/parallel/quantized_linear.py:168-176), for batched decode
// (16-32 rows), short prefill chunks and the vocab-sharded lm_head over a batch of
// last positions (transformer.py:466-475).  Here the product is bandwidth-bound or
// close to the ridge (4 M flops per W4 weight byte), so the kernel is built around
// the weight stream rather than around MFMA tiles:
//
// * A workgroup owns BN = 32 x (consumer waves) weight rows over a K range (one K
//   split) and all M rows of x (MT blocks of 32).  Each consumer wave owns 32 weight
//   rows: the B operand of v_mfma_f32_32x32x16_bf16, shared by the MT x blocks (the A
//   operands), so every weight is dequantized once per workgroup.
// * Four producer waves issue every LDS-DMA (global_load_lds_dwordx4) and do nothing
//   else, so an issue that waits for room in the CU's memory queue stalls only them.
//   (Measured on the 64-row lm_head: the stream alone, with the consumers idle, takes
//   34 us with four producers and 46 us with two; the consumers' arithmetic alone
//   takes 49 us, so the arithmetic, not the stream, now bounds the kernel.)
// * K advances one quantization group (64) per stage; one barrier per stage.  Three
//   LDS rings, each fed ahead of use:
//     x       one stage (32 MT rows x 128 B) per slot, NX slots;
//     codes   one "item" of IG groups (128 B of every weight row: 4 groups W4, 2 W8)
//             per slot, 3 slots, loaded in IG pieces with the x stages (a weight row's
//             bytes arrive as whole 128-byte lines, not as 32-byte pieces of lines);
//     s, b    the 8 groups' scales and biases of the BN rows, 2 block slots.
//   Every stage's DMA list has the same length per producer, so each producer waits
//   for its part of stage g with one vmcnt immediate; the barrier then publishes the
//   stage and frees the slots the previous stage read.
// * Dequant in registers.  Above 32 rows: bf16(s q + b), one fp32 FMA per weight (the
//   GEMM's rule).  Up to 32 rows (one x block): the decode GEMVs' rule, exact codes on
//   MFMA and the group's scale and bias applied to its fp32 sums (s P + b S), so that
//   a decode batch rounds as a single sequence does.  The k order inside a group is
//   permuted so that a lane's codes of the 4 MFMA k-steps are one 16-byte LDS read
//   (W4): lane half h, step ks holds k = 32 h + 8 ks + e; x rows use the same order
//   (16-byte chunk 4 h + ks).
// * Rows are XOR-swizzled in 16-byte chunks (x by row, codes by row / 2), so the
//   operand reads are free of LDS bank conflicts; the DMA writes lanes in order, so
//   each lane loads the chunk that belongs at its position.
// * With one K split the tile is rounded to bf16 and written (bias after rounding);
//   with several, each split writes fp32 partials and the split-K pass sums them in
//   split order (deterministic).
#include "dma_util.h"

#include "../../include/shardcompute_hip.h"

#include <type_traits>
#include <utility>

namespace sc {

struct BandArgs {
    const uint16_t *x;
    const uint8_t *wq;      // packed codes, rows of K * bits / 8 bytes
    const uint16_t *s;
    const uint16_t *b;
    const uint16_t *bias;
    uint16_t *y;
    float *partials;        // [ksplit, M, N] fp32, or null: y is written directly
    int M, N, K, G;
    int gps;                // groups per K split (a multiple of 8)
};

namespace band {

using namespace dma;

constexpr int NP = 4;                                  // producer waves
constexpr int LDS_CAP = 160 * 1024;

// bytes of an x stage: 32 mt rows (mt = 0: 16 rows) of 64 bf16
__host__ __device__ constexpr int band_xb(int mt) { return mt == 0 ? 2048 : mt * 4096; }
// The rings' slots: nx x stages and ns code items.  The stream's rate is the bytes in
// flight, nx - 2 stages' lists, so the pair with the most x slots that fits is taken:
// * the code ring's refill must not overtake its readers (x runs lx = nx - 1 stages ahead;
//   an item is loaded over the ig stages of the item before it): lx <= ig (ns - 2) + 1;
// * a scale/bias block's refill must not overtake its one read: lx <= 7;
// * 4-wave workgroups of up to 32 rows stay within half the LDS, two to a CU;
// * W8 above 32 rows keeps 3 code items: with 5 (two to three times the bytes in flight)
//   its first stage starts later and a 45-row product of any size took 1.3 us longer.
// 4 items where 3 were: 45 rows W4, 4096 -> 6144 16.3 -> 14.9 us, 14336 -> 4096 22.4 -> 19.4.
struct Rings {
    int nx, ns;
};
__host__ __device__ constexpr Rings band_rings(int bits, int mt, int nw) {
    const int cap = mt <= 1 && nw == 4 ? 80 * 1024 : LDS_CAP;
    const int ig = bits == 4 ? 4 : 2, item = 32 * nw * 128;
    Rings best{0, 3};
    for (int ns = 3; ns <= (bits == 8 && mt >= 2 ? 3 : 6); ++ns) {
        int nx = (cap - ns * item - 2 * (1024 * nw)) / band_xb(mt);
        if (nx > ig * (ns - 2) + 2) nx = ig * (ns - 2) + 2;
        if (nx > 8) nx = 8;
        if (nx > best.nx) best = Rings{nx, ns};
    }
    return best;
}

template <int BITS, int MT, int NW>
struct Geo {
    static constexpr int BN = 32 * NW;                 // weight rows per workgroup
    static constexpr int XB = band_xb(MT);             // x stage: 32 MT (or 16) rows x 64 bf16
    static constexpr int WROW = BITS == 4 ? 32 : 64;   // bytes of one weight row per group
    static constexpr int IG = 128 / WROW;              // groups per code item
    static constexpr int WIB = BN * 128;               // code item bytes
    static constexpr int SBB = 2 * BN * 16;            // scales then biases, 8 groups of BN rows
    static constexpr int NX = band_rings(BITS, MT, NW).nx;   // x ring slots
    static constexpr int NS = band_rings(BITS, MT, NW).ns;   // code ring slots
    static constexpr int LX = NX - 1;                  // stages the x DMA runs ahead
    static constexpr int O_W = NX * XB;                // LDS: x ring, code ring, s/b slots
    static constexpr int O_SB = O_W + NS * WIB;
    static constexpr int LDS = O_SB + 2 * SBB;
    static constexpr int XI = XB / 1024;               // DMA instructions per stage: x,
    static constexpr int WPI = WIB / 1024 / IG;        // a piece of a code item,
    static constexpr int TI = WPI + 1 + XI;            // one scale/bias instruction
    static constexpr int DP = (TI + NP - 1) / NP;      // per producer: DP or DP - 1
    static constexpr int NFULL = TI % NP == 0 ? NP : TI % NP;   // producers issuing DP
    static constexpr int THREADS = 64 * (NW + NP);
    static_assert(NX >= 3 && LX <= IG * (NS - 2) + 1 && LX <= 7, "rings");
    static_assert(LDS <= LDS_CAP, "LDS");
    static_assert((LX - 1) * DP < 64, "vmcnt range");
};

// stage(number of lists issued after it, false, its index) for the last sizeof...(Is) stages
template <class F, int... Is>
__device__ __forceinline__ void tail_stages(F &&stage, int g, std::integer_sequence<int, Is...>) {
    constexpr int L = (int)sizeof...(Is);
    (stage(std::integral_constant<int, L - 1 - Is>{}, false, g + Is), ...);
}

}  // namespace band

using namespace band;

// Up to 16 rows (MT = 0): the consumers' loop, by the rule of the 17-32-row one below (exact
// codes on MFMA, y += s P + (b - 128 s) S in fp32) at half its work:
// * 16x16x32 MFMAs on two blocks of 16 weight rows: half the MFMA time, x operands and
//   scale FMAs of a 32-row block;
// * (b - 128 s) S is one fp32 MFMA per block and group: A holds each lane's own part of the
//   row's x sum (v_dot2 with ones over the operands it has), B the column's b - 128 s in
//   every k slot, so the contraction adds the parts up, instead of a second bf16 MFMA
//   chain with all-ones weights and 4 more FMAs.  (Summing a group's x in one wave and
//   sharing it through LDS is less work still, but as a branch of the unrolled stages it
//   doubled the registers.)
// Measured with its split-K pass, this and the shorter tail of the stream (us, 16 rows,
// before -> after): W4 4096 -> 6144 11.9 -> 10.8, 14336 -> 4096 17.5 -> 16.3, 8192 -> 7168
// 17.8 -> 16.0, 3584 -> 8192 12.4 -> 11.3; W8 12.8 -> 12.3, 20.6 -> 19.9, 19.8 -> 19.6, 14.1 -> 13.7.
template <int BITS, int NW>
__device__ __forceinline__ void consume16(const BandArgs &a, uint8_t *smem, int wave, int lane, int n0, int nb,
                                          int split) {
    using C = Geo<BITS, 0, NW>;
    constexpr int NX = C::NX, IG = C::IG;
    const int li = lane & 15, lq = lane >> 4;          // operand row (column), k part
    uint32_t nib16 = 0x000F000Fu, magic = 0x43004300u; // opaque: one v_and_or_b32 per code pair
    asm volatile("" : "+s"(nib16));
    asm volatile("" : "+v"(magic));
    f32x4_t acc[2] = {f32x4_t{}, f32x4_t{}};
    // lane part lq's k-step ks takes k chunk 2 lq + ks of the group (8 k), for x and codes
    // alike, so that a lane's codes of the group are contiguous
    uint32_t xo[2], wo[2];
    int wsw[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
        xo[ks] = (uint32_t)(li * 128 + (((2 * lq + ks) ^ (li & 7) ^ ((li >> 3) & 1)) << 4));
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int rr = 32 * wave + 16 * c + li;
        wo[c] = (uint32_t)(C::O_W + rr * 128);
        wsw[c] = (rr >> 1) & 7;
    }
    uint4 sv[2], bv[2];                                // scales, biases of the block's 8 groups
    int xslot = 0, wslot = 0;
    for (int bk = 0; bk < nb; ++bk) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            __syncthreads();                           // stage 8 bk + j landed
            if (j == 0) {
                const uint8_t *sb = smem + C::O_SB + (bk & 1) * C::SBB;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    sv[c] = *reinterpret_cast<const uint4 *>(sb + 16 * (32 * wave + 16 * c + li));
                    bv[c] = *reinterpret_cast<const uint4 *>(sb + 16 * (C::BN + 32 * wave + 16 * c + li));
                }
            }
            const uint8_t *xs = smem + xslot * C::XB;
            const uint8_t *ws = smem + wslot * C::WIB;
            const int gi = j % IG;                     // group of the code item
            uint4 xv[2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) xv[ks] = *reinterpret_cast<const uint4 *>(xs + xo[ks]);
            uint32_t w[2][BITS == 4 ? 2 : 4];          // the lane's codes of the group
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if constexpr (BITS == 4) {
                    const uint2 v = *reinterpret_cast<const uint2 *>(
                        ws + wo[c] + ((((2 * gi + (lq >> 1)) ^ wsw[c]) << 4) | ((lq & 1) << 3)));
                    w[c][0] = v.x; w[c][1] = v.y;
                } else {
                    const uint4 v = *reinterpret_cast<const uint4 *>(ws + wo[c] + (((4 * gi + lq) ^ wsw[c]) << 4));
                    w[c][0] = v.x; w[c][1] = v.y; w[c][2] = v.z; w[c][3] = v.w;
                }
            }
            f32x4_t P[2] = {f32x4_t{}, f32x4_t{}};
            float sx = 0.f;                            // this lane's part of the group's x sum
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                sx = add_pair_bf16(xv[ks].x, sx);
                sx = add_pair_bf16(xv[ks].y, sx);
                sx = add_pair_bf16(xv[ks].z, sx);
                sx = add_pair_bf16(xv[ks].w, sx);
                const bf16x8_t A = as_bf16x8(BITS == 4 ? perm_w4x(xv[ks]) : xv[ks]);
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    bf16x8_t B;
                    if constexpr (BITS == 4) {
                        const uint32_t v = w[c][ks];
                        B = as_bf16x8(and_or(v, nib16, magic), and_or(v >> 4, nib16, magic),
                                      and_or(v >> 8, nib16, magic), and_or(v >> 12, nib16, magic));
                    } else {
                        const uint32_t w0 = w[c][2 * ks], w1 = w[c][2 * ks + 1];
                        B = as_bf16x8(byte_pair_lo(w0), byte_pair_hi(w0), byte_pair_lo(w1), byte_pair_hi(w1));
                    }
                    P[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, P[c], 0, 0, 0);
                }
            }
            // the compiler leaves no wait states between a v_dot2 and the MFMA that reads its
            // result (the last terms of the sum were missing): 4 here
            asm volatile("s_nop 3" : "+v"(sx));
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float sf = bf2f(wh(sv[c], j)), bf = bf2f(wh(bv[c], j));
                acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx, BITS == 4 ? fmaf(-128.f, sf, bf) : bf, acc[c], 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[c][r] = fmaf(sf, P[c][r], acc[c][r]);
            }
            xslot = xslot + 1 == NX ? 0 : xslot + 1;
            if (j % IG == IG - 1) wslot = wslot + 1 == C::NS ? 0 : wslot + 1;
        }
    }

    // lane (column li, part lq) register r holds row 4 lq + r
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int n = n0 + 32 * wave + 16 * c + li;
        if (n >= a.N) continue;
        const float bb = (!a.partials && a.bias) ? bf2f(a.bias[n]) : 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = 4 * lq + r;
            if (m >= a.M) continue;
            if (a.partials) {
                a.partials[((size_t)split * a.M + m) * a.N + n] = acc[c][r];
            } else {
                uint32_t o = f2bf(acc[c][r]);
                if (a.bias) o = f2bf(bf2f(o) + bb);
                a.y[(size_t)m * a.N + n] = (uint16_t)o;
            }
        }
    }
}

// The LDS holds one workgroup per CU, so (NW + NP) / 4 waves share a SIMD.  With 8 x
// blocks the compiler, left to aim for more waves, keeps the accumulators and x
// operands in fewer registers and serialises each MFMA behind its LDS read; told the
// real occupancy it prefetches them (160 rows: 38.5 -> 32.3 us on a 4096 x 6144
// product).  The smaller blocks measured no faster with it.
template <int BITS, int MT, int NW>
__global__ void __launch_bounds__(64 * (NW + NP))
__attribute__((amdgpu_waves_per_eu((NW + NP + 3) / 4, MT >= 8 ? (NW + NP + 3) / 4 : 8)))
qgemm_band_kernel(BandArgs a) {
    using C = Geo<BITS, MT, NW>;
    constexpr int NX = C::NX, LX = C::LX, IG = C::IG;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = a.M, N = a.N;
    const int n0 = blockIdx.x * C::BN;
    const int split = blockIdx.y;
    const int g0 = split * a.gps;
    const int ng = min(a.G - g0, a.gps);               // groups of this split, a multiple of 8
    const int nb = ng >> 3;                            // scale/bias blocks
    const int ni = ng / IG;                            // code items
    const size_t row_bytes = (size_t)a.K * BITS / 8;

    if (wave >= NW) {
        // ================================================================ producers
        // Stage t's list: the code piece (t - 1) % IG of item (t - 1) / IG + 1 (item j's
        // last piece rides with stage IG j, so waiting for stage IG j's x covers it),
        // the scale/bias instruction t % 8 of block t / 8 + 1 (repeats of the last
        // instruction when the block has fewer than 8; block b's last rides with stage
        // 8b - 1), then the x stage.  Instruction i goes to producer i % NP.  Items,
        // blocks and stages past the split are clamped: the reloads rewrite slots nobody reads any
        // more (or the same bytes), and keep the lists' lengths equal.
        const int pw = wave - NW;
        const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
        const uint8_t *xbase = reinterpret_cast<const uint8_t *>(a.x) + (size_t)g0 * 128;
        const uint8_t *wbase = a.wq + (size_t)n0 * row_bytes + (size_t)g0 * C::WROW;
        // per-lane offsets, the same for every stage
        // x instruction q: rows 8q + lane / 8, position p = lane % 8 holds chunk p ^ swz(row)
        auto xoff = [&](int q) -> uint32_t {
            const int xr = 8 * q + (lane >> 3);
            const int c = (lane & 7) ^ (xr & 7) ^ ((xr >> 3) & 1);
            return (uint32_t)((min(xr, M - 1) * a.K + 8 * c) * 2);
        };
        // code instruction q of an item: rows 8q + lane / 8, position p holds chunk p ^ (row / 2 % 8)
        auto woff = [&](int q) -> uint32_t {
            const int wr = 8 * q + (lane >> 3);
            const int c = (lane & 7) ^ ((wr >> 1) & 7);
            return (uint32_t)((size_t)(min(n0 + wr, N - 1) - n0) * row_bytes + 16 * c);
        };
        auto issue_sb = [&](int u, int blk) __attribute__((always_inline)) {
            // chunks [64 u, 64 u + 64) of [scales BN | biases BN]: instructions u < NW / 2
            // are scales, the rest biases
            const bool is_b = u >= NW / 2;
            const int row = min(n0 + 64 * u + lane - (is_b ? C::BN : 0), N - 1) - n0;
            const uint8_t *base =
                reinterpret_cast<const uint8_t *>((is_b ? a.b : a.s) + (size_t)n0 * a.G + g0 + 8 * blk);
            dma16s(base, (uint32_t)(row * a.G * 2), lds0 + C::O_SB + (blk & 1) * C::SBB + 1024 * u);
        };
        auto issue_w = [&](int item, int q) __attribute__((always_inline)) {
            // instruction q of code item `item` (clamped to the split) into its slot
            const int ic = min(item, ni - 1);
            dma16s(wbase + (size_t)ic * 128, woff(q), lds0 + C::O_W + (item % C::NS) * C::WIB + 1024 * q);
        };
        auto issue = [&](int t) __attribute__((always_inline)) {
            const int tc = min(t, ng - 1);
            const int item = (t + IG - 1) / IG, piece = (t + IG - 1) % IG;     // (t - 1) / IG + 1, (t - 1) % IG
            const uint32_t xs = lds0 + (t % NX) * C::XB;
#pragma unroll
            for (int r = 0; r < C::DP; ++r) {
                const int i = pw + r * NP;
                if (i < C::WPI) issue_w(item, piece * C::WPI + i);
                else if (i == C::WPI) issue_sb(min(t & 7, NW - 1), min((t >> 3) + 1, nb - 1));
                else if (i < C::TI) dma16s(xbase + (size_t)tc * 128, xoff(i - C::WPI - 1), xs + 1024 * (i - C::WPI - 1));
            }
        };
        // prologue: code item 0 (all but its last piece, which rides with stage 0),
        // scale/bias block 0, stages 0 .. LX - 1
        for (int q = pw; q < (IG - 1) * C::WPI; q += NP) issue_w(0, q);
        for (int u = pw; u < NW; u += NP) issue_sb(u, 0);
        for (int t = 0; t < LX; ++t) issue(t);
        auto stage = [&](auto after, bool more, int g) __attribute__((always_inline)) {
            // this producer's part of stage g (and everything it issued before) landed; `after`
            // lists were issued since
            constexpr int n = decltype(after)::value;
            if (pw < C::NFULL) wait_vm<n * C::DP>();
            else wait_vm<n * (C::DP - 1)>();
            __syncthreads();                                // stage g visible; slots of g - 1 free
            if (more) issue(g + LX);
        };
        // The last LX stages (ng >= 8 > LX) have nothing left to issue: reloads of the last
        // stage in their place (up to half a split's bytes again) cost 3-8 % of a product.
        // Not so for W8 above 32 rows, where the two loops are 0.6 % slower than the reloads
        // of its three lists (45 x 8192 -> 7168: 21.7 against 21.8 us).
        constexpr bool TAIL = BITS == 4 || MT <= 1;
        int g = 0;
        for (; g < (TAIL ? ng - LX : ng); ++g) stage(std::integral_constant<int, LX - 1>{}, true, g);
        if constexpr (TAIL) tail_stages(stage, g, std::make_integer_sequence<int, LX>{});
        wait_vm<0>();                                       // no DMA may land after the workgroup ends
        return;
    }

    // ==================================================================== consumers
    const int li = lane & 31, h = lane >> 5;
    const int rr = 32 * wave + li;                     // this lane's weight row in the tile
    if constexpr (MT == 0) {
        consume16<BITS, NW>(a, smem, wave, lane, n0, nb, split);
        return;
    }
    uint32_t nib = 0x0F0F0F0Fu;                        // opaque: one v_cvt_f32_ubyteN per code
    asm volatile("" : "+s"(nib));
    uint32_t nib16 = 0x000F000Fu, magic = 0x43004300u; // opaque: one v_and_or_b32 per code pair
    asm volatile("" : "+s"(nib16));
    asm volatile("" : "+v"(magic));
    constexpr int MB = MT > 1 ? MT : 1;
    f32x16_t acc[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[i] = f32x16_t{};
    // x operand (row 32 i + li, 16-byte chunk 4 h + ks) of a stage
    auto xoff = [&](int i, int ks) -> uint32_t {
        const int r = 32 * i + li;
        return (uint32_t)(r * 128 + ((((4 * h + ks) ^ (r & 7) ^ ((r >> 3) & 1))) << 4));
    };
    const int wsw = (rr >> 1) & 7;                     // this row's chunk swizzle in a code item
    auto compute = [&](int xslot, int wslot, int gi, int j, uint4 sv, uint4 bv) __attribute__((always_inline)) {
        const uint8_t *xs = smem + xslot * C::XB;
        const uint8_t *ws = smem + C::O_W + wslot * C::WIB + rr * 128;
        const float sf = bf2f(wh(sv, j)), bf = bf2f(wh(bv, j));
        uint4 wv0, wv1;
        if (BITS == 4) {       // group gi = chunks 2 gi, 2 gi + 1; this lane's half h
            wv0 = *reinterpret_cast<const uint4 *>(ws + 16 * ((2 * gi + h) ^ wsw));
            wv1 = wv0;
        } else {               // group gi = chunks 4 gi .. 4 gi + 3; this lane's two
            wv0 = *reinterpret_cast<const uint4 *>(ws + 16 * ((4 * gi + 2 * h) ^ wsw));
            wv1 = *reinterpret_cast<const uint4 *>(ws + 16 * ((4 * gi + 2 * h + 1) ^ wsw));
        }
        if constexpr (MT == 1) {
            // Up to 32 rows: the decode GEMVs' rule (qgemv_m1_kernel, qgemv16_kernel),
            // so a batch computes as one sequence does: the MFMAs take the exact codes
            // (W4: 128 + q in bf16, slots [q0 q4 q1 q5 q2 q6 q3 q7], x permuted alike;
            // W8: q), a second MFMA chain with all-ones weights sums the group's x, and
            // y += s * P + (b - 128 s) * S (W8: b * S) in fp32.
            const uint32_t ones = 0x3F803F80u;
            const bf16x8_t B1 = as_bf16x8(ones, ones, ones, ones);
            f32x16_t P = f32x16_t{}, S = f32x16_t{};
            uint4 xn = *reinterpret_cast<const uint4 *>(xs + xoff(0, 0));
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                uint4 xv = xn;
                if (ks + 1 < 4) xn = *reinterpret_cast<const uint4 *>(xs + xoff(0, ks + 1));
                bf16x8_t B;
                if (BITS == 4) {
                    xv = perm_w4x(xv);
                    const uint32_t w = wc(wv0, ks);
                    B = as_bf16x8(and_or(w, nib16, magic), and_or(w >> 4, nib16, magic),
                                  and_or(w >> 8, nib16, magic), and_or(w >> 12, nib16, magic));
                } else {
                    const uint4 v = ks < 2 ? wv0 : wv1;
                    const uint32_t w0 = wc(v, 2 * (ks & 1)), w1 = wc(v, 2 * (ks & 1) + 1);
                    B = as_bf16x8(byte_pair_lo(w0), byte_pair_hi(w0), byte_pair_lo(w1), byte_pair_hi(w1));
                }
                P = mfma32x32x16(as_bf16x8(xv), B, P);
                S = mfma32x32x16(as_bf16x8(xv), B1, S);
            }
            const float cf = BITS == 4 ? fmaf(-128.f, sf, bf) : bf;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[0][r] = fmaf(sf, P[r], fmaf(cf, S[r], acc[0][r]));
            return;
        }
        // x operands one k-step ahead of the MFMAs that use them
        uint4 xa[2][MB];
#pragma unroll
        for (int i = 0; i < MB; ++i) xa[0][i] = *reinterpret_cast<const uint4 *>(xs + xoff(i, 0));
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            if (ks + 1 < 4) {
#pragma unroll
                for (int i = 0; i < MB; ++i)
                    xa[(ks + 1) & 1][i] = *reinterpret_cast<const uint4 *>(xs + xoff(i, ks + 1));
            }
            bf16x8_t B;
            if (BITS == 4) {
                const uint32_t w = wc(wv0, ks);
                const uint32_t lo = w & nib, hi = (w >> 4) & nib;       // codes 0 2 4 6 / 1 3 5 7
                B = as_bf16x8(cvt_pk_bf16(fmaf(sf, ubyte_f32(lo, 0), bf), fmaf(sf, ubyte_f32(hi, 0), bf)),
                              cvt_pk_bf16(fmaf(sf, ubyte_f32(lo, 1), bf), fmaf(sf, ubyte_f32(hi, 1), bf)),
                              cvt_pk_bf16(fmaf(sf, ubyte_f32(lo, 2), bf), fmaf(sf, ubyte_f32(hi, 2), bf)),
                              cvt_pk_bf16(fmaf(sf, ubyte_f32(lo, 3), bf), fmaf(sf, ubyte_f32(hi, 3), bf)));
            } else {
                const uint4 v = ks < 2 ? wv0 : wv1;
                const uint32_t w0 = wc(v, 2 * (ks & 1)), w1 = wc(v, 2 * (ks & 1) + 1);
                B = as_bf16x8(cvt_pk_bf16(fmaf(sf, ubyte_f32(w0, 0), bf), fmaf(sf, ubyte_f32(w0, 1), bf)),
                              cvt_pk_bf16(fmaf(sf, ubyte_f32(w0, 2), bf), fmaf(sf, ubyte_f32(w0, 3), bf)),
                              cvt_pk_bf16(fmaf(sf, ubyte_f32(w1, 0), bf), fmaf(sf, ubyte_f32(w1, 1), bf)),
                              cvt_pk_bf16(fmaf(sf, ubyte_f32(w1, 2), bf), fmaf(sf, ubyte_f32(w1, 3), bf)));
            }
#pragma unroll
            for (int i = 0; i < MB; ++i) acc[i] = mfma32x32x16(as_bf16x8(xa[ks & 1][i]), B, acc[i]);
        }
    };

    int xslot = 0, wslot = 0;
    for (int bk = 0; bk < nb; ++bk) {
        uint4 sv = make_uint4(0u, 0u, 0u, 0u), bv = sv;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            __syncthreads();                          // stage 8 bk + j landed
            if (j == 0) {
                const uint8_t *sb = smem + C::O_SB + (bk & 1) * C::SBB;
                sv = *reinterpret_cast<const uint4 *>(sb + 16 * rr);
                bv = *reinterpret_cast<const uint4 *>(sb + 16 * (C::BN + rr));
            }
            compute(xslot, wslot, j % IG, j, sv, bv);
            xslot = xslot + 1 == NX ? 0 : xslot + 1;
            if (j % IG == IG - 1) wslot = wslot + 1 == C::NS ? 0 : wslot + 1;
        }
    }

    // ---- epilogue: lane (column li, half h) register r holds row 8 (r / 4) + 4 h + r % 4
    // of each 32-row block
    const int n = n0 + rr;
    if (n < N) {
        const float bb = (!a.partials && a.bias) ? bf2f(a.bias[n]) : 0.f;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
                if (m < M) {
                    if (a.partials) {
                        a.partials[((size_t)split * M + m) * N + n] = acc[i][r];
                    } else {
                        uint32_t o = f2bf(acc[i][r]);
                        if (a.bias) o = f2bf(bf2f(o) + bb);
                        a.y[(size_t)m * N + n] = (uint16_t)o;
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------- host side

template <int BITS, int MT, int NW>
static int launch_band_t(const BandArgs &a, int tiles, int ksplit, hipStream_t stream) {
    using C = Geo<BITS, MT, NW>;
    if (device_info().max_lds_per_block < C::LDS) return set_error(SC_EUNSUPPORTED, "qgemm_band: LDS too small");
    auto kern = qgemm_band_kernel<BITS, MT, NW>;
    static bool configured = false;
    if (!configured) {
        SC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS));
        configured = true;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)ksplit), dim3(C::THREADS), C::LDS, stream, a);
    SC_HIP_CHECK(hipGetLastError());
    return SC_OK;
}

// 8 consumer waves (256 rows per workgroup) up to 64 rows of x; 4 above (the 32-row
// blocks' accumulators need the larger register budget of 6-wave workgroups)
template <int BITS, int MT>
static int launch_band_mt(const BandArgs &a, int nw, int tiles, int ksplit, hipStream_t stream) {
    if constexpr (MT <= 2) {
        if (nw == 8) return launch_band_t<BITS, MT, 8>(a, tiles, ksplit, stream);
    }
    return launch_band_t<BITS, MT, 4>(a, tiles, ksplit, stream);
}

// LDS bytes of a variant (Geo<>::LDS)
static int band_lds(int bits, int mt, int nw) {
    const Rings r = band_rings(bits, mt, nw);
    return r.nx * band_xb(mt) + r.ns * (32 * nw * 128) + 2 * (1024 * nw);
}

static int band_mt(int M) { return M <= 16 ? 0 : M <= 32 ? 1 : M <= 64 ? 2 : M <= 128 ? 4 : 8; }

struct BandPlan {
    int nw, tiles, ksplit, bps;                          // bps: scale/bias blocks per split
};

// 8-wave workgroups (256 rows) unless too few tiles would be left to fill the CUs even
// with every scale/bias block a split of its own (twice over above 32 rows, three quarters
// over up to 32: measured on the decode shapes); then the K splits that bring the
// workgroups to about one round (two per CU for the small 4-wave ones).
static BandPlan plan_band(int M, int N, int K, int bits, int force_nw, int force_split) {
    const int mt = band_mt(M), nb = K / 512;
    const int P = device_info().num_cus;
    BandPlan p;
    p.nw = force_nw ? force_nw : 8;
    if (!force_nw && (long)((N + 255) / 256) * nb < (mt <= 1 ? 3L * P / 4 : 2L * P)) p.nw = 4;
    if (mt > 2) p.nw = 4;
    p.tiles = (N + 32 * p.nw - 1) / (32 * p.nw);
    const int per_cu = band_lds(bits, mt, p.nw) <= 80 * 1024 ? 2 : 1;
    int ks = force_split ? force_split : (int)((P * per_cu + p.tiles / 2) / p.tiles);
    if (ks < 1) ks = 1;
    if (ks > nb) ks = nb;
    p.bps = (nb + ks - 1) / ks;
    p.ksplit = (nb + p.bps - 1) / p.bps;
    return p;
}

// Returns SC_EUNSUPPORTED when the shape does not suit this kernel (the caller falls
// back).  force_nw / force_split (0 = automatic) pin the plan for measurements.
// no_alloc: the split-K partials go to the allocation-free scratch array (shapes that
// need more are SC_EUNSUPPORTED) instead of the library-owned buffer.
// swiglu_half > 0: the weight is gate|up stacked (N = 2 swiglu_half) and y
// [M, swiglu_half] receives silu(gate) * up, applied by the split-K pass.  K in one piece
// needs no scratch and no fp32 partials: the product goes to gate_up [M, N] (16-byte
// aligned) and the activation reads it (8B gate|up with it, W4, at
// 100 and 160 rows 48.5 and 76.2 us through partials, 46.6 and 73.6 so).
// keep (plain products): the partials are left to the caller's pass (keep->splits > 0)
// instead of being summed into y.
int launch_qgemm_band(const uint16_t *x, const uint32_t *wq, const uint16_t *s, const uint16_t *b,
                      const uint16_t *bias, uint16_t *y, int M, int N, int K, int bits, hipStream_t stream,
                      bool no_alloc, int swiglu_half, int force_nw, int force_split, SplitKeep *keep,
                      uint16_t *gate_up) {
    if (M < 1 || M > 256 || N < 1) return SC_EUNSUPPORTED;
    if (bits != 4 && bits != 8) return SC_EUNSUPPORTED;
    if (K % 512) return SC_EUNSUPPORTED;                 // whole 8-group scale/bias blocks
    if (swiglu_half && N != 2 * swiglu_half) return SC_EUNSUPPORTED;
    if (((uintptr_t)x % 16) || ((uintptr_t)wq % 16) || ((uintptr_t)s % 16) || ((uintptr_t)b % 16))
        return SC_EUNSUPPORTED;
    // per-lane DMA offsets are 32-bit: x rows (M K 2 bytes) and a tile's weight rows
    if ((long long)M * K * 2 >= (1LL << 31) || (long long)K >= (1LL << 23)) return SC_EUNSUPPORTED;
    const int mt = band_mt(M), G = K / 64;
    int nw = force_nw ? force_nw : 8;
    if (nw != 4 && nw != 8) return set_error(SC_EINVAL, "qgemm_band: waves %d (4 or 8)", nw);
    const BandPlan p = plan_band(M, N, K, bits, force_nw, force_split);
    nw = p.nw;
    const int tiles = p.tiles, ksplit = p.ksplit, bps = p.bps;

    BandArgs a;
    a.x = x; a.wq = reinterpret_cast<const uint8_t *>(wq); a.s = s; a.b = b; a.bias = bias; a.y = y;
    a.partials = nullptr;
    a.M = M; a.N = N; a.K = K; a.G = G; a.gps = 8 * bps;
    const bool then_act = swiglu_half && ksplit == 1 && gate_up && (uintptr_t)y % 16 == 0;
    const bool with_partials = ksplit > 1 || (swiglu_half && !then_act);
    if (then_act) a.y = gate_up;
    if (with_partials) {
        const size_t need = (size_t)ksplit * M * N;
        if (no_alloc) {
            if (need * sizeof(float) > (size_t)SC_QMM_NOALLOC_SCRATCH_BYTES) return SC_EUNSUPPORTED;
            const int rc = qmm_noalloc_scratch(&a.partials);
            if (rc) return rc;
        } else {
            SplitKScratch ws;
            const int rc = splitk_scratch(need, 1, &ws);
            if (rc) return rc;
            a.partials = ws.partials;
        }
    }
    int rc;
    if (bits == 4) {
        rc = mt == 0 ? launch_band_mt<4, 0>(a, nw, tiles, ksplit, stream)
           : mt == 1 ? launch_band_mt<4, 1>(a, nw, tiles, ksplit, stream)
           : mt == 2 ? launch_band_mt<4, 2>(a, nw, tiles, ksplit, stream)
           : mt == 4 ? launch_band_mt<4, 4>(a, nw, tiles, ksplit, stream)
                     : launch_band_mt<4, 8>(a, nw, tiles, ksplit, stream);
    } else {
        rc = mt == 0 ? launch_band_mt<8, 0>(a, nw, tiles, ksplit, stream)
           : mt == 1 ? launch_band_mt<8, 1>(a, nw, tiles, ksplit, stream)
           : mt == 2 ? launch_band_mt<8, 2>(a, nw, tiles, ksplit, stream)
           : mt == 4 ? launch_band_mt<8, 4>(a, nw, tiles, ksplit, stream)
                     : launch_band_mt<8, 8>(a, nw, tiles, ksplit, stream);
    }
    if (rc) return rc;
    if (then_act) return launch_silu_mul(gate_up, M, swiglu_half, y, stream);
    if (keep) {
        keep->partials = with_partials ? a.partials : nullptr;
        keep->splits = with_partials ? ksplit : 0;
        if (with_partials && !swiglu_half) return SC_OK;
    }
    if (with_partials) return launch_qmm_finalize(a.partials, ksplit, M, N, bias, y, swiglu_half, stream);
    return SC_OK;
}

}  // namespace sc
