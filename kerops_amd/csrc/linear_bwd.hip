// Backward of the pointwise (1x1x1) ReLU-linear op on the matrix cores (gfx950), one pass over x and grad:
//
//   dx[v, ci] = (x[v, ci] > 0) ? fp16( sum_co g[v, co] * Wm[ci, co] ) : 0
//   dW[ci, co] = sum_v relu(x[v, ci]) * g[v, co]                          (fp32 end to end)
//
// x is [V][CIN] fp16, g is [V][COUT] fp16 (the memory of channels_last_3d tensors), Wm is [CIN][COUT] fp16.
// The op moves 2*V*(2*CIN + COUT) bytes: it is HBM-bound; both products run on v_mfma_f32_32x32x16_f16 so
// that the arithmetic stays a fraction of the memory time.
//
// A workgroup of four wavefronts loops over tiles of 64 to 256 voxels (lb_tile).  The tile of x and of g is staged
// through LDS (global -> registers one tile ahead -> LDS, rows of 16-byte chunks).
//  * dx is computed transposed, dx^T[ci, v] = Wm[ci, :] . g^T[:, v]: the A operand is a 32-row block of Wm
//    (16-byte fragments pre-arranged in LDS), the B operand is one 16-byte chunk of a voxel's g row.  One
//    (32 voxels x 32 input channels) block per wavefront; the fp32 result is rounded to fp16, bounced through
//    an LDS tile and written back as 16-byte chunks with the (x > 0) mask applied from the staged x tile.
//  * dW[ci, co] reduces over voxels, which is the slow axis of both operands in memory: the fragments
//    "8 consecutive voxels of one channel" are gathered from the LDS tiles with transposing reads (two
//    ds_read_b64_tr_b16 per fragment, see SwizzledRows in common.hpp; the ReLU is
//    applied to the x fragment in registers).  The (32 x 32) output blocks are distributed over the
//    wavefronts (with fewer than four blocks the wavefronts split the voxels instead) and accumulated in
//    fp32 registers over all tiles of the workgroup; at the end every workgroup writes its partial
//    [CIN][COUT] matrix to the workspace and a second kernel adds them in a fixed order (deterministic).
//    A matrix instruction rounds its running sum twice, from a zero accumulator a little downwards (2e-9 on average, inputs
//    ~ N(0, 1)).  Against the first, a block has two or more accumulators that take the voxel steps in turn; they and the
//    sums of wavefronts that split the voxels are added in fp64 and rounded once for the row.  Against the second, odd
//    workgroups work on -g and -Wm (the same bits of dx) and return minus their sum.  Relative error of dW against 64 bits,
//    with one accumulator and fp32 sums of the split / now: 0.9 M voxels 16 -> 16 170e-9 / 94e-9, 64 -> 64 258e-9 /
//    183e-9, 128 -> 128 268e-9 / 116e-9, at 1 % more time.
#include "common.hpp"

namespace kerops {

typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kLbThreads = 256;
constexpr int kLbWaves = kLbThreads / kWave;

// Voxels per tile.  A tile's loads are all a workgroup has in flight, two to four workgroups run on a compute unit, and
// the memory system needs about 40 KB in flight per compute unit: 64 voxels, 128 where the rows are short.  us with 64 /
// 128 voxels and the best workgroup count of each: 16 -> 64 at 0.9 M voxels 36.1 / 34.8, 16 -> 16 at 4 M 74.4 / 66.2
// (256 voxels: 69.1), 32 -> 32 at 4 M 125.9 / 133.5, 64 -> 16 at 4096 6.1 / 6.7.
// The AFFINE kernel has the registers of two workgroups on a compute unit and takes the tiles that fill them (16 -> 16 at
// 4 M voxels 75.4 with 256, 83.1 with 128; 32 -> 32 140.4 with 128, 156.5 with 64 and three workgroups; 77.0 and 140.8 with
// the sums as they are now).
constexpr int lb_tile(int cin, int cout, bool affine)
{
    if (affine) return cin + cout >= 96 ? 64 : cin + cout >= 48 ? 128 : 256;
    return (cin == 16 && cout <= 64) || (cin == 32 && cout == 16) ? 128 : 64;
}

template <int CIN, int COUT, bool AFFINE>
struct LbCfg {
    static constexpr int TILE = lb_tile(CIN, COUT, AFFINE);
    static constexpr int MTI = (CIN + 31) / 32, MTO = (COUT + 31) / 32;  // 32-channel blocks
    static constexpr int KSO = COUT / 16;                                 // k steps of the dx product
    static constexpr int KSV = TILE / 16;                                 // k steps (voxels) of the dW product
    static constexpr int XP = CIN, GP = COUT, DP = CIN;  // dense rows (halves); swizzled: SwizzledRows / BounceTile in common.hpp
    static constexpr int NVT = TILE / 32;                                  // 32-voxel blocks
    static constexpr int NBD = NVT * MTI;                                 // dx blocks (32 voxels x 32 channels) per tile
    static constexpr int NBW = MTI * MTO;                                 // dW blocks
    static constexpr int KSPL = NBW >= kLbWaves ? 1 : kLbWaves / NBW;     // voxel split when blocks are few
    static constexpr int BPW = NBW >= kLbWaves ? NBW / kLbWaves : 1;      // dW blocks per wavefront
    static constexpr int STEPS = KSV / KSPL;                               // voxel steps of a wavefront per tile and block
    // Accumulators of a block.  128 -> 128 has registers for one: it starts a chain from zero in every tile.
    static constexpr bool TILE_CHAIN = BPW == 4;
    static constexpr int NSET = TILE_CHAIN ? 1 : KSPL == 4 && STEPS > 2 ? STEPS : 2;
    static constexpr int NXC = TILE * CIN / 8, NGC = TILE * COUT / 8;  // 16-byte chunks per tile
    static constexpr int NLX = (NXC + kLbThreads - 1) / kLbThreads, NLG = (NGC + kLbThreads - 1) / kLbThreads;
    static constexpr int XS_OFF = 0;
    static constexpr int GS_OFF = XS_OFF + TILE * XP * 2;
    static constexpr int DS_OFF = GS_OFF + TILE * GP * 2;
    static constexpr int WL_OFF = (DS_OFF + TILE * DP * 2 + 15) / 16 * 16;
    static constexpr int TILE_BYTES = WL_OFF + MTI * KSO * 64 * 16;
    static constexpr int SPLIT_BYTES = KSPL > 1 ? KSPL * CIN * COUT * 8 : 0;  // the sums of the split, after the last tile
    static constexpr int LDS_BYTES = TILE_BYTES > SPLIT_BYTES ? TILE_BYTES : SPLIT_BYTES;
    static_assert(CIN % 16 == 0 && CIN <= 128 && COUT % 16 == 0 && COUT <= 128, "channels in {16,32,64,128}");
    static_assert(NBW % kLbWaves == 0 || kLbWaves % NBW == 0, "blocks divide over the wavefronts");
    static_assert(KSV % KSPL == 0, "voxel steps divide over the split");
    static_assert(LDS_BYTES >= kLbWaves * 2 * CIN * 8, "the sums of scale and shift fit the tiles' LDS");
};

// eight fp16 values (a float) with flipped signs where `signs` (0x80008000 or 0) says so
__device__ __forceinline__ half8_t flip_signs(const half8_t& h, uint32_t signs)
{
    return __builtin_bit_cast(half8_t, __builtin_bit_cast(u32x4_t, h) ^ signs);
}

__device__ __forceinline__ float flip_sign(float f, uint32_t signs)
{
    return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, f) ^ (signs & 0x80000000u));
}

// Sums over a wavefront's tiles of 2 x 8 values per lane, lane l holding the channels 8 (l % CGI) + 0..7.  A tile's values
// of the four lanes l % 16 + {0, 16, 32, 48} are added in fp32 by two rounds of lane swaps that also deal the 16 sums out
// to these lanes, four each; the tiles are added in fp64.  8 registers per lane where fp32 sums of all values take 16, and
// no chain over the tiles (at 128 channels and 0.9 M voxels: relative error of dscale 140e-9 with the chain).
template <int CGI>
struct ChannelSums {
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    static __device__ __forceinline__ float swap32_add(float a, float b)  // lanes below 32: sum of a, the others: of b
    {
        const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                        false, false);
        return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
    }
    static __device__ __forceinline__ float swap16_add(float a, float b)  // even rows of 16 lanes: sum of a, odd ones: of b
    {
        const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                        false, false);
        return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
    }
    __device__ __forceinline__ void add(const float (&v)[2][8])
    {
        float w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = swap32_add(v[0][k], v[1][k]);
#pragma unroll
        for (int k = 0; k < 4; ++k) sum[k] += (double)swap16_add(w[k], w[k + 4]);
    }
    __device__ __forceinline__ void store(double* dst)  // dst[2][8 CGI]
    {
        const int lane = threadIdx.x % kWave, row = lane / 16;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
            for (int off = 8; off >= CGI; off >>= 1) sum[k] += __shfl_xor(sum[k], off, 64);
            if (lane % 16 < CGI) dst[(row / 2) * 8 * CGI + (lane % CGI) * 8 + 4 * (row % 2) + k] = sum[k];
        }
    }
};

// AFFINE: the op's input is z = fp16(max(fma(x, scale[c], shift[c]), 0)), formed from the loaded x on its way to LDS, and
// the gradient goes on through that map where it leaves: with gz the fp16 gradient of z that the plain kernel would
// store, gm = x * scale > -shift ? gz : 0, dx = fp16(scale * gm), dscale = sum x * gm, dshift = sum gm (the arithmetic of
// the batch-norm + ReLU stream ops, same bits for dx).  A thread stages and writes back the same chunks of a tile, so
// the raw x it needs again stays in its registers, and all its chunks have the same eight channels.  Neither z nor gz
// reach memory: 3 tensors are moved instead of 8 (16 -> 16 channels at 2.1 M voxels 42 us, 100 as bnrelu_fwd,
// relu_linear_bwd and bnrelu_bwd).
template <int CIN, int COUT, bool AFFINE>
__global__ __launch_bounds__(kLbThreads, 2) void relu_linear_bwd_kernel(const half_t* __restrict__ x,
                                                                        const half_t* __restrict__ g,
                                                                        const half_t* __restrict__ Wm,
                                                                        half_t* __restrict__ dx, float* __restrict__ ws,
                                                                        int64_t V, const float* __restrict__ scale,
                                                                        const float* __restrict__ shift, int drain)
{
    constexpr int CGI = CIN / 8, ROW = CIN * COUT + (AFFINE ? 2 * CIN : 0);  // ROW: floats of a row of the workspace
    using Cfg = LbCfg<CIN, COUT, AFFINE>;
    constexpr int XP = Cfg::XP, GP = Cfg::GP, DP = Cfg::DP, KSO = Cfg::KSO, KSV = Cfg::KSV;
    constexpr int NLX = Cfg::NLX, NLG = Cfg::NLG, BPW = Cfg::BPW, KSPL = Cfg::KSPL;
    __shared__ __attribute__((aligned(16))) unsigned char smem[Cfg::LDS_BYTES];
    unsigned char* xs = smem + Cfg::XS_OFF;
    unsigned char* gs = smem + Cfg::GS_OFF;
    using XT = SwizzledRows<CIN>;
    using GT = SwizzledRows<COUT>;
    half_t* ds = reinterpret_cast<half_t*>(smem + Cfg::DS_OFF);
    half8_t* wl = reinterpret_cast<half8_t*>(smem + Cfg::WL_OFF);

    const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
    const int il = lane % 32, hl = lane / 32;
    const half8_t z8 = {0, 0, 0, 0, 0, 0, 0, 0};

    const uint32_t signs = blockIdx.x % 2 ? 0x80008000u : 0u;

    // A fragments of the dx product: wl[(mt*KSO + s)*64 + lane] = Wm[32 mt + il][16 s + 8 hl + 0..7].  Loaded here, all at
    // once, and written to LDS behind the first tile's loads: one trip to memory for both.
    constexpr int NWL = Cfg::MTI * KSO * 64, NLW = (NWL + kLbThreads - 1) / kLbThreads;
    const plane_rsrc_t wr = plane_rsrc(Wm, CIN * COUT * 2);
    half8_t wpre[NLW];
#pragma unroll
    for (int k = 0; k < NLW; ++k) {
        const int i = t + k * kLbThreads, l = i % 64, s = (i / 64) % KSO, mt = i / (64 * KSO);
        // (rows past CIN, of a 16-channel block's upper half, are past the matrix: zeros)
        wpre[k] = plane_load16<false>(wr, (uint32_t)(((32 * mt + l % 32) * COUT + 16 * s + 8 * (l / 32)) * 2));
    }

    // this wavefront's dW blocks (mi, ni) and its share of the voxel steps
    const int wb0 = Cfg::NBW >= kLbWaves ? wave : wave % Cfg::NBW;
    const int kpart = Cfg::NBW >= kLbWaves ? 0 : wave / Cfg::NBW;
    float16_t wacc[BPW][Cfg::NSET];
#pragma unroll
    for (int bb = 0; bb < BPW; ++bb)
#pragma unroll
        for (int n = 0; n < Cfg::NSET; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) wacc[bb][n][i] = 0.0f;
    int ndone = 0;  // tiles of this workgroup

    // dscale and dshift: this thread's values of FLUSH tiles (a chain of 8, 4 at 128 channels), and all of them
    constexpr int FLUSH = (CIN == 128 ? 4 : 8) / NLX;
    float sc[AFFINE ? 8 : 1], sh[AFFINE ? 8 : 1], aacc[2][8];
    ChannelSums<CGI> asum;
    auto clear_affine = [&]() {
#pragma unroll
        for (int k = 0; k < 8; ++k) aacc[0][k] = aacc[1][k] = 0.0f;
    };
    if constexpr (AFFINE) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            sc[j] = scale[(t % CGI) * 8 + j];
            sh[j] = shift[(t % CGI) * 8 + j];
        }
        clear_affine();
    }

    const int64_t ntiles = (V + Cfg::TILE - 1) / Cfg::TILE;
    // The tile's part of a tensor with `row` bytes per voxel: nothing stands behind a condition and the wait for a tile's
    // loads leaves the stores of the one before in flight (us with the conditions / now: 64 -> 64 at 0.05 / 0.9 M voxels 14.2 / 13.2, 66.5 / 64.3, with the batch-norm map at 0.9 M 77.8 / 73.0;
    // 128 -> 128 at 0.05 / 0.3 M 29.6 / 27.4, 60.9 / 56.5).
    auto tile_rsrc = [&](const half_t* p, int64_t tile, int row) {
        return rows_rsrc(p, tile * Cfg::TILE, Cfg::TILE, V, row);
    };
    half8_t xpre[NLX], gpre[NLG];
    auto prefetch = [&](int64_t tile) {  // (chunks past the tile: zeros)
        const plane_rsrc_t xr = tile_rsrc(x, tile, 2 * CIN), gr = tile_rsrc(g, tile, 2 * COUT);
#pragma unroll
        for (int j = 0; j < NLX; ++j) xpre[j] = plane_load16<true>(xr, (uint32_t)(t + j * kLbThreads) * 16);
#pragma unroll
        for (int j = 0; j < NLG; ++j) gpre[j] = plane_load16<true>(gr, (uint32_t)(t + j * kLbThreads) * 16);
    };

    int64_t tile = blockIdx.x;
    prefetch(tile);
#pragma unroll
    for (int j = 0; j < NLX; ++j) plane_store16<true>(plane_rsrc(dx, 0u), 0u, z8);  // (of nothing: as many as a tile's)
#pragma unroll
    for (int k = 0; k < NLW; ++k)
        if (t + k * kLbThreads < NWL) wl[t + k * kLbThreads] = flip_signs(wpre[k], signs);
    for (; tile < ntiles; tile += gridDim.x) {
        const int64_t v0 = tile * Cfg::TILE;
        half8_t xraw[AFFINE ? NLX : 1];
        if (!AFFINE && drain) wait_all_accesses();  // (uniform)
        // ---- stage the tile (rows past V are zero: they add nothing to dW) ----
#pragma unroll
        for (int j = 0; j < NLX; ++j) {
            const int c = t + j * kLbThreads;
            half8_t z = xpre[j];
            if constexpr (AFFINE) {
                xraw[j] = xpre[j];
                const bool inside = v0 + c / CGI < V;  // the map of a row past V is not zero
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    z[k] = inside ? (half_t)fmaxf(__builtin_fmaf((float)xpre[j][k], sc[k], sh[k]), 0.0f) : (half_t)0;
            }
            if (c < Cfg::NXC) *reinterpret_cast<half8_t*>(xs + XT::chunk16(c / CGI, c % CGI)) = z;
        }
#pragma unroll
        for (int j = 0; j < NLG; ++j) {
            const int c = t + j * kLbThreads;
            if (c < Cfg::NGC)
                *reinterpret_cast<half8_t*>(gs + GT::chunk16(c / (COUT / 8), c % (COUT / 8))) = flip_signs(gpre[j], signs);
        }
        __syncthreads();
        prefetch(tile + gridDim.x);

        // ---- dx^T blocks: (vt, mt) = 32 voxels x 32 input channels ----
#pragma unroll (Cfg::TILE_CHAIN && AFFINE ? 1 : 8)  // (128 -> 128: unrolled, it spills registers)
        for (int bd = 0; bd < (Cfg::NBD + kLbWaves - 1) / kLbWaves; ++bd) {
            const int blk = wave + bd * kLbWaves;
            if (blk < Cfg::NBD) {  // wavefront-uniform
                const int vt = blk % Cfg::NVT, mt = blk / Cfg::NVT;
                // chunk 2 s + hl of the lane's voxel row: the swizzle is an XOR, so step s is the offset of step 0 ^ 32 s
                const int grow = GT::chunk16(32 * vt + il, hl);
                float16_t acc;
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
                for (int s = 0; s < KSO; ++s) {
                    const half8_t bfrag = *reinterpret_cast<const half8_t*>(gs + (grow ^ (32 * s)));
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(wl[(mt * KSO + s) * 64 + lane], bfrag, acc, 0, 0, 0);
                }
                // acc[i]: input channel 32 mt + 8 (i/4) + 4 hl + i%4 of voxel 32 vt + il
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    const int ci = 32 * mt + 8 * gq + 4 * hl;
                    if (ci < CIN) {
                        half4_t o;
#pragma unroll
                        for (int jj = 0; jj < 4; ++jj) o[jj] = (half_t)acc[4 * gq + jj];
                        *reinterpret_cast<half4_t*>(reinterpret_cast<unsigned char*>(ds) + BounceTile<CIN>::piece(32 * vt + il, 4 * mt + gq, hl)) = o;
                    }
                }
            }
        }

        // ---- dW blocks: A = relu(x)^T (channel il of 8 consecutive voxels), B = g likewise ----
        float16_t chain;  // TILE_CHAIN: the tile's sum of the block before, added behind the next block's instructions
        auto add_chain = [&](int bb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                wacc[bb][0][i] += chain[i];
                // (added here: left alone, the compiler keeps the chains of all blocks and adds them at the tile's end)
                asm volatile("" : "+v"(wacc[bb][0][i]));
            }
        };
#pragma unroll
        for (int bb = 0; bb < BPW; ++bb) {
            const int blk = wb0 + bb * kLbWaves;
            const int mi = blk / Cfg::MTO, ni = blk % Cfg::MTO;
            int xoff[2], goff[2];  // transposing reads: lane = channel 32 mi + il / 32 ni + il, registers = 8 voxels
            XT::tr_offsets(lane, mi, xoff);
            GT::tr_offsets(lane, ni, goff);
            auto step = [&](int sp, float16_t c) {
                const int s = kpart + sp * KSPL;
                const half8_t af = __builtin_elementwise_max(XT::read_tr(xs, xoff, s), z8);  // relu(x), packed
                return __builtin_amdgcn_mfma_f32_32x32x16_f16(af, GT::read_tr(gs, goff, s), c, 0, 0, 0);
            };
            if constexpr (Cfg::TILE_CHAIN) {  // (AFFINE has no registers for a second chain)
                float16_t next;
#pragma unroll
                for (int i = 0; i < 16; ++i) next[i] = 0.0f;
#pragma unroll
                for (int sp = 0; sp < Cfg::STEPS; ++sp) next = step(sp, next);
                if (!AFFINE && bb > 0) add_chain(bb - 1);
                chain = next;
                if constexpr (AFFINE) add_chain(bb);
            } else if constexpr (Cfg::STEPS == 1) {
                if (ndone % 2) wacc[bb][1] = step(0, wacc[bb][1]);
                else wacc[bb][0] = step(0, wacc[bb][0]);
            } else {
#pragma unroll
                for (int sp = 0; sp < Cfg::STEPS; ++sp) wacc[bb][sp % Cfg::NSET] = step(sp, wacc[bb][sp % Cfg::NSET]);
            }
        }
        if constexpr (Cfg::TILE_CHAIN && !AFFINE) add_chain(BPW - 1);
        ++ndone;
        __syncthreads();

        // ---- dx write-back: 16-byte chunks, masked by x > 0 (rows past V are staged as zeros) ----
        if constexpr (AFFINE && FLUSH == 1) clear_affine();
        const plane_rsrc_t dr = tile_rsrc(dx, tile, 2 * CIN);
#pragma unroll
        for (int j = 0; j < NLX; ++j) {
            const int c = t + j * kLbThreads;
            const int row = c / (CIN / 8), cc = c % (CIN / 8);
            half8_t o = z8;
            if (c < Cfg::NXC) {
                const half8_t xv = *reinterpret_cast<const half8_t*>(xs + XT::chunk16(row, cc));
                o = BounceTile<CIN>::read(reinterpret_cast<const unsigned char*>(ds), row, cc);
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) o[jj] = xv[jj] > (half_t)0 ? o[jj] : (half_t)0;
                if constexpr (AFFINE) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const float xf = (float)xraw[j][k];
                        const float gm = __fmul_rn((float)o[k], (__fmul_rn(xf, sc[k]) > -sh[k]) ? 1.0f : 0.0f);
                        o[k] = (half_t)as_fp32_value(__fmul_rn(sc[k], gm));
                        aacc[0][k] = __builtin_fmaf(xf, gm, aacc[0][k]);
                        aacc[1][k] += gm;
                    }
                }
            }
            plane_store16<true>(dr, (uint32_t)c * 16, o);
        }
        if constexpr (AFFINE) {
            if (ndone % FLUSH == 0) {
                asum.add(aacc);
                if constexpr (FLUSH > 1) clear_affine();
            }
        }
        __syncthreads();
    }

    // ---- partial dW of this workgroup: row blockIdx of the workspace, [CIN][COUT] fp32 (AFFINE: and [2][CIN]) ----
    // Wavefronts that split the voxels add their sums in LDS first (the tiles are done: the loop ends in a barrier).
    float* out = ws + (int64_t)blockIdx.x * ROW;
    double* part = reinterpret_cast<double*>(smem) + kpart * (CIN * COUT);
#pragma unroll
    for (int bb = 0; bb < BPW; ++bb) {
        const int blk = wb0 + bb * kLbWaves;
        const int mi = blk / Cfg::MTO, ni = blk % Cfg::MTO;
        const int co = 32 * ni + il;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int ci = 32 * mi + 8 * (i / 4) + 4 * hl + i % 4;
            if (ci >= CIN || co >= COUT) continue;
            if constexpr (KSPL > 1) {
                double sum = wacc[bb][0][i];
#pragma unroll
                for (int n = 1; n < Cfg::NSET; ++n) sum += (double)wacc[bb][n][i];
                part[ci * COUT + co] = sum;
            } else {
                out[ci * COUT + co] = flip_sign(Cfg::NSET > 1 ? wacc[bb][0][i] + wacc[bb][Cfg::NSET - 1][i] : wacc[bb][0][i], signs);
            }
        }
    }
    if constexpr (KSPL > 1) {
        __syncthreads();
        const double* all = reinterpret_cast<const double*>(smem);
        for (int j = t; j < CIN * COUT; j += kLbThreads) {
            double sum = all[j];
#pragma unroll
            for (int k = 1; k < KSPL; ++k) sum += all[k * (CIN * COUT) + j];
            out[j] = flip_sign((float)sum, signs);
        }
    }
    if constexpr (AFFINE) {
        if constexpr (KSPL > 1) __syncthreads();  // the LDS sums have been read
        double* red = reinterpret_cast<double*>(smem);
        if constexpr (FLUSH > 1) asum.add(aacc);
        asum.store(red + wave * 2 * CIN);
        __syncthreads();
        if (t < 2 * CIN) {
            double sum = 0.0;
#pragma unroll
            for (int wv = 0; wv < kLbWaves; ++wv) sum += red[wv * 2 * CIN + t];
            out[CIN * COUT + t] = (float)sum;
        }
    }
}

// Workgroups per compute unit (the AFFINE kernel: two).  Two: what the LDS holds at 128 -> 128 channels, and a third only adds a row to the
// partial sums (64 -> 128 at 0.35 M voxels: 43.4 us with two, 47.7 with three; 128 -> 128 at 0.26 M: 54.8 and 67.7).
// 16 -> 16 has the fewest bytes in flight and the shortest rows of sums and takes four.  In volumes of half a million
// voxels and more, where the rows of sums are few against the tiles, three pay at 32 -> 32 (0.2 M voxels 13.7 us with
// two, 14.5 with three; 0.9 M 36.9 and 34.8; 15.7 M 523 and 492) and 16 -> 128 (0.2 M 19.1 and 19.7; 0.9 M 57.6 and
// 55.4; with stores left in flight 4 M 217 and 224, but the sums of two are longer by half, which costs bits), and 16 -> 16
// has one more than it needs (4 M: 68.9 with four, 66.2 with three).
static int lb_blocks(int64_t V, int cin, int cout, bool affine)
{
    const bool narrow = cin == 16 && cout == 16 && !affine;
    int per_cu = narrow ? 4 : 2;
    if (V >= (1 << 19) && !affine && (narrow || (cin == 32 && cout == 32) || (cin == 16 && cout == 128))) per_cu = 3;
    const int64_t ntiles = ceil_div64(V, lb_tile(cin, cout, affine));
    return (int)std::max<int64_t>(1, std::min<int64_t>(ntiles, per_cu * device_geometry().cus));
}

// Voxels from which a wavefront of the plain kernel waits for its stores before it goes on.  Large volumes run at the memory's rate,
// and then some pairs are the fastest where a workgroup reads and writes in turns, as it did with a condition around every
// store (us without / with the wait: 16 -> 16 at 4 M voxels 66.4 / 66.0, 30 M 501 / 474; 16 -> 32 at 16 M 332 / 326; 16 -> 64 at 4 M
// 135 / 130, 16 M 538 / 514; 32 -> 16 at 16 M 454 / 449; 32 -> 32 at 4 M 129 / 125, 16 M 526 / 490; 32 -> 64 at 16 M 677 / 666;
// 32 -> 128 at 4 M 268 / 257; 64 -> 32 at 4 M 214 / 213, 16 M 898 / 878; 64 -> 128 at 12 M 1086 / 1033), others are not (16 -> 32
// at 4 M 84.8 / 87.1, 16 -> 128 at 4 M 224 / 227, 64 -> 64 at 16 M 1083 / 1089, 128 -> 64 at 8 M 911 / 954).  Behind other ops a
// launch without the wait can be the faster one where in a row of its own it is not: 64 -> 128 behind the forward op, both,
// at 0.9 M 169 / 172, 2 M 367 / 377, 4 M 743 / 753 (alone 350 / 336), 6 M 1142 / 1140, 8 M 1567 / 1540; the other pairs gain or
// are equal there too (32 -> 128 at 2 M 329 / 323, 32 -> 32 at 4 M 254 / 250, 16 -> 64 at 4 M 326 / 320).
static constexpr int64_t lb_drain_from(int cin, int cout)
{
    constexpr int64_t kVoxels = 1000;
    if (cin == 128 || (cin == 64 && cout < 128 && cout != 32) || (cin == 16 && cout == 128)) return INT64_MAX;
    if (cout == 2 * cin && cin <= 32) return 12000 * kVoxels;
    if ((cin == 32 && cout == 16) || (cin == 64 && cout == 128)) return 6000 * kVoxels;
    if ((cin == 16 && cout == 16) || (cin == 64 && cout == 32)) return 3000 * kVoxels;
    return cout == 128 ? 700 * kVoxels : 2000 * kVoxels;  // 32 -> 128; 16 -> 64, 32 -> 32
}

// daffine: the AFFINE kernel's [2][CIN] sums, null without scale and shift
template <int CIN, int COUT>
static int launch_lb(const half_t* x, const float* scale, const float* shift, const half_t* g, const half_t* Wm,
                     half_t* dx, void* dW, int dw_dtype, float* daffine, float* ws, int64_t V, hipStream_t s)
{
    const int blocks = lb_blocks(V, CIN, COUT, scale != nullptr), drain = V >= lb_drain_from(CIN, COUT);
    if (scale)
        hipLaunchKernelGGL((relu_linear_bwd_kernel<CIN, COUT, true>), dim3(blocks), dim3(kLbThreads), 0, s, x, g, Wm, dx,
                           ws, V, scale, shift, drain);
    else
        hipLaunchKernelGGL((relu_linear_bwd_kernel<CIN, COUT, false>), dim3(blocks), dim3(kLbThreads), 0, s, x, g, Wm,
                           dx, ws, V, scale, shift, drain);
    int rc = check_launch("relu_linear_bwd");
    if (rc != KEROPS_OK) return rc;
    const int ncols = CIN * COUT + (scale ? 2 * CIN : 0);
    if (dw_dtype == KEROPS_DTYPE_F16)
        launch_reduce_rows_f16(ws, blocks, ncols, (half_t*)dW, daffine, CIN * COUT, s);
    else
        launch_reduce_rows(ws, blocks, ncols, (float*)dW, daffine, CIN * COUT, 1.0, s);
    return check_launch("relu_linear_bwd_reduce");
}

}  // namespace kerops

using namespace kerops;

static bool lb_channels_ok(int c) { return c == 16 || c == 32 || c == 64 || c == 128; }

static int64_t lb_workspace(const char* op, int64_t V, int Cin, int Cout, bool affine)
{
    if (V <= 0) {
        set_error("%s: non-positive size", op);
        return KEROPS_E_BADARG;
    }
    if (!lb_channels_ok(Cin) || !lb_channels_ok(Cout)) {
        set_error("%s: built for Cin, Cout in {16,32,64,128} (got %d -> %d)", op, Cin, Cout);
        return KEROPS_E_UNSUPPORTED_C;
    }
    return (int64_t)lb_blocks(V, Cin, Cout, affine) * (Cin * Cout + (affine ? 2 * Cin : 0)) * (int64_t)sizeof(float);
}

static int lb_run(const char* op, const void* x, const float* scale, const float* shift, const void* g, const void* Wm,
                  void* dx, void* dW, int32_t dw_dtype, float* daffine, void* workspace, int64_t workspace_bytes,
                  int64_t V, int32_t Cin, int32_t Cout, void* stream)
{
    if (!grad_dtype_ok(dw_dtype)) {
        set_error("%s: dw_dtype must be KEROPS_DTYPE_F32 or KEROPS_DTYPE_F16", op);
        return KEROPS_E_BADARG;
    }
    const int64_t need = lb_workspace(op, V, Cin, Cout, daffine != nullptr);
    if (need < 0) return (int)need;
    if (!x || !g || !Wm || !dx || !dW || !aligned16(x) || !aligned16(g) || !aligned16(Wm) || !aligned16(dx)) {
        set_error("%s: null or misaligned pointer", op);
        return KEROPS_E_BADARG;
    }
    if (!workspace || !aligned16(workspace) || workspace_bytes < need) {
        set_error("%s: workspace of %lld bytes required, %lld given", op, (long long)need, (long long)workspace_bytes);
        return KEROPS_E_WORKSPACE;
    }
    const half_t* xh = (const half_t*)x;
    const half_t* gh = (const half_t*)g;
    const half_t* wh = (const half_t*)Wm;
    hipStream_t s = (hipStream_t)stream;
#define KEROPS_LB_CASE(CI, CO)    \
    if (Cin == CI && Cout == CO)  \
        return launch_lb<CI, CO>(xh, scale, shift, gh, wh, (half_t*)dx, dW, dw_dtype, daffine, (float*)workspace, V, s);
    KEROPS_LB_CASE(16, 16)
    KEROPS_LB_CASE(16, 32)
    KEROPS_LB_CASE(16, 64)
    KEROPS_LB_CASE(16, 128)
    KEROPS_LB_CASE(32, 16)
    KEROPS_LB_CASE(32, 32)
    KEROPS_LB_CASE(32, 64)
    KEROPS_LB_CASE(32, 128)
    KEROPS_LB_CASE(64, 16)
    KEROPS_LB_CASE(64, 32)
    KEROPS_LB_CASE(64, 64)
    KEROPS_LB_CASE(64, 128)
    KEROPS_LB_CASE(128, 16)
    KEROPS_LB_CASE(128, 32)
    KEROPS_LB_CASE(128, 64)
    KEROPS_LB_CASE(128, 128)
#undef KEROPS_LB_CASE
    set_error("%s: no kernel for %d -> %d", op, Cin, Cout);
    return KEROPS_E_UNSUPPORTED_C;
}

extern "C" int64_t kerops_relu_linear_bwd_workspace_bytes(int64_t V, int32_t Cin, int32_t Cout)
{
    return lb_workspace("relu_linear_bwd", V, Cin, Cout, false);
}

extern "C" int kerops_relu_linear_bwd_f16(const void* x, const void* g, const void* Wm, void* dx, float* dW,
                                          void* workspace, int64_t workspace_bytes, int64_t V, int32_t Cin,
                                          int32_t Cout, void* stream)
{
    return kerops_relu_linear_bwd_f16_out(x, g, Wm, dx, dW, KEROPS_DTYPE_F32, workspace, workspace_bytes, V, Cin, Cout,
                                          stream);
}

extern "C" int kerops_relu_linear_bwd_f16_out(const void* x, const void* g, const void* Wm, void* dx, void* dW,
                                              int32_t dw_dtype, void* workspace, int64_t workspace_bytes, int64_t V,
                                              int32_t Cin, int32_t Cout, void* stream)
{
    return lb_run("relu_linear_bwd", x, nullptr, nullptr, g, Wm, dx, dW, dw_dtype, nullptr, workspace, workspace_bytes, V,
                  Cin, Cout, stream);
}

extern "C" int64_t kerops_bnrelu_linear_bwd_workspace_bytes(int64_t V, int32_t Cin, int32_t Cout)
{
    return lb_workspace("bnrelu_linear_bwd", V, Cin, Cout, true);
}

extern "C" int kerops_bnrelu_linear_bwd_f16(const void* x, const float* scale, const float* shift, const void* g,
                                            const void* Wm, void* dx, void* dW, int32_t dw_dtype, float* daffine,
                                            void* workspace, int64_t workspace_bytes, int64_t V, int32_t Cin,
                                            int32_t Cout, void* stream)
{
    if (!scale || !shift || !daffine) {
        set_error("bnrelu_linear_bwd: null scale, shift or daffine");
        return KEROPS_E_BADARG;
    }
    return lb_run("bnrelu_linear_bwd", x, scale, shift, g, Wm, dx, dW, dw_dtype, daffine, workspace, workspace_bytes, V,
                  Cin, Cout, stream);
}
