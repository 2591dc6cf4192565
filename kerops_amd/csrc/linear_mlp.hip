// Inverted-bottleneck pointwise block on the matrix cores (gfx950):
//
//   hid[v, :] = relu( fp16(x[v, :] @ Wup) + bias )      (fp16 add, C -> 2C channels)
//   out[v, :] = fp16( hid[v, :] @ Wdown ) + add[v, :]   (fp16 add, 2C -> C channels)
//
// x, add, out are [V][C] fp16 (the memory of channels_last_3d tensors), Wup [C][2C], Wdown [2C][C], bias [2C].
// The op moves 6*V*C bytes; the hidden activation never leaves the registers.
//
// Each wavefront owns tiles of 32 voxels and computes both products transposed on v_mfma_f32_32x32x16_f16
// (A = rows of W^T, pre-arranged 16-byte fragments in LDS; B = the voxel's channel vector).  The first
// product leaves lane (v, h) with the hidden channels 32 mt + 8 gq + 4 h + 0..3 of voxel v; since the
// reduction index of the second product may be enumerated in any order as long as both operands agree, its
// k step (mt, gp) takes exactly the 8 values the lane already holds for gq = 2 gp, 2 gp + 1, and the
// fragments of Wdown^T are arranged in the same order.  The result is bounced through a wavefront-private
// LDS tile and written back as 16-byte chunks with the fp16 residual add fused in.
#include "common.hpp"

namespace kerops {

typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kMlpThreads = 256;
constexpr int kMlpWaves = kMlpThreads / kWave;

template <int C>
struct MlpCfg {
    static constexpr int HID = 2 * C;
    static constexpr int MT1 = HID / 32;        // 32-row blocks of hidden channels
    static constexpr int KS1 = C / 16;          // k steps of the first product
    static constexpr int MO = (C + 31) / 32;    // 32-row blocks of output channels
    static constexpr int KS2 = HID / 16;        // k steps of the second product: (mt, gp)
    static constexpr int RH = C;                // output tile: dense rows, swizzled (BounceTile in common.hpp)
    static constexpr int A1_OFF = 0;
    static constexpr int A2_OFF = A1_OFF + MT1 * KS1 * 64 * 16;
    static constexpr int B_OFF = A2_OFF + MO * KS2 * 64 * 16;
    static constexpr int T_OFF = (B_OFF + HID * 2 + 15) / 16 * 16;
    static constexpr int LDS_BYTES = T_OFF + kMlpWaves * 32 * RH * 2;
    static_assert(C == 16 || C == 32 || C == 64, "C in {16,32,64}");
};

template <int C>
__global__ __launch_bounds__(kMlpThreads) void lin_brelu_lin_add_kernel(const half_t* __restrict__ x,
                                                                        const half_t* __restrict__ Wup,
                                                                        const half_t* __restrict__ Wdown,
                                                                        const half_t* __restrict__ bias,
                                                                        const half_t* __restrict__ add,
                                                                        half_t* __restrict__ out, int64_t V)
{
    using Cfg = MlpCfg<C>;
    constexpr int HID = Cfg::HID, MT1 = Cfg::MT1, KS1 = Cfg::KS1, MO = Cfg::MO, KS2 = Cfg::KS2, RH = Cfg::RH;
    __shared__ __attribute__((aligned(16))) unsigned char smem[Cfg::LDS_BYTES];
    half_t* a1 = reinterpret_cast<half_t*>(smem + Cfg::A1_OFF);
    half_t* a2 = reinterpret_cast<half_t*>(smem + Cfg::A2_OFF);
    half_t* bs = reinterpret_cast<half_t*>(smem + Cfg::B_OFF);

    const int t = threadIdx.x, lane = t % kWave, wave = __builtin_amdgcn_readfirstlane(t / kWave);
    const int vl = lane % 32, hl = lane / 32;

    // a1[((mt*KS1 + s)*64 + l)*8 + j] = Wup[16 s + 8 (l/32) + j][32 mt + l%32]
    // a2[((mo*KS2 + s)*64 + l)*8 + j] = Wdown[hidden channel of (s = 2 mt + gp, l/32, j)][32 mo + l%32]
    // All their loads are in flight at once and go to LDS behind the first tile's (the weights need not be aligned: two bytes
    // each).  One after the other, ahead of the tile, they cost C = 32 at 20000
    // voxels 1.9 us of 5.9, C = 64 at 5000 0.8 of 8.6.
    constexpr int N1 = MT1 * KS1 * 512 / kMlpThreads, N2 = MO * KS2 * 512 / kMlpThreads;
    static_assert(HID <= kMlpThreads, "a bias value per thread");
    half_t w1[N1], w2[N2];
#pragma unroll
    for (int k = 0; k < N1; ++k) {
        const int i = t + k * kMlpThreads, j = i % 8, l = (i / 8) % 64, s = (i / 512) % KS1, mt = i / (512 * KS1);
        w1[k] = Wup[(16 * s + 8 * (l / 32) + j) * HID + 32 * mt + l % 32];
    }
#pragma unroll
    for (int k = 0; k < N2; ++k) {
        const int i = t + k * kMlpThreads, j = i % 8, l = (i / 8) % 64, s = (i / 512) % KS2, mo = i / (512 * KS2);
        const int mt = s / 2, gp = s % 2;
        const int ch = 32 * mt + 8 * (2 * gp + j / 4) + 4 * (l / 32) + j % 4;
        const int co = 32 * mo + l % 32;
        const half_t w = Wdown[ch * C + co % C];
        w2[k] = co < C ? w : (half_t)0;
    }
    const half_t bias_t = bias[t % HID];

    const half8_t* a1f = reinterpret_cast<const half8_t*>(a1) + lane;
    const half8_t* a2f = reinterpret_cast<const half8_t*>(a2) + lane;
    unsigned char* my = smem + Cfg::T_OFF + wave * 32 * RH * 2;
    using Tile = BounceTile<C>;

    const int64_t ntiles = (V + 31) / 32;
    const int64_t tiles_per_round = (int64_t)gridDim.x * kMlpWaves;
    const int64_t nrounds = (ntiles + tiles_per_round - 1) / tiles_per_round;
    // Loads of a tile: x fragments, and residual chunks in the order in which the results leave the LDS tile.  Those of the
    // next tile are issued as soon as this tile has used the registers, so that both streams are in flight while the
    // results are stored; loaded where they are used, a tile waits for memory twice (C = 64 at 0.1 M voxels 28.2 us, 18.0
    // early, C = 32 9.0 and 7.8).  Nothing stands behind a condition (rows_rsrc), so a tile waits for its own loads and
    // leaves the stores of the one before in flight (C = 16 at 0.9 M voxels 17.4 -> 16.2 us).
    constexpr int NC = 32 * C / 8 / kWave;
    half8_t xb[KS1], ab[NC];
    auto load_x = [&](int64_t tidx) {
        const plane_rsrc_t r = rows_rsrc(x, tidx * 32, 32, V, 2 * C);
        // rows of 128 bytes need the cache to hold the line until the row's other loads arrive
#pragma unroll
        for (int s = 0; s < KS1; ++s) xb[s] = plane_load16<(C <= 32)>(r, (uint32_t)(vl * 2 * C + 32 * s + 16 * hl));
    };
    const int64_t first = (int64_t)blockIdx.x * kMlpWaves + wave;
    load_x(first);
    {
        // (with the loads and stores in the order of the loop, stores of nothing: the waits are the same on both ways in)
        const plane_rsrc_t ar = rows_rsrc(add, first * 32, 32, V, 2 * C);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            plane_store16<true>(plane_rsrc(out, 0u), 0u, half8_t{});
            ab[k] = plane_load16<true>(ar, (uint32_t)(k * kWave + lane) * 16);
        }
    }
#pragma unroll
    for (int k = 0; k < N1; ++k) a1[t + k * kMlpThreads] = w1[k];
#pragma unroll
    for (int k = 0; k < N2; ++k) a2[t + k * kMlpThreads] = w2[k];
    if (t < HID) bs[t] = bias_t;
    __syncthreads();
    for (int64_t r = 0; r < nrounds; ++r) {
        const int64_t tidx = (r * gridDim.x + blockIdx.x) * kMlpWaves + wave;
        {
            // ---- first product, bias, ReLU: the B fragments of the second product ----
            half8_t hb[KS2];
#pragma unroll
            for (int mt = 0; mt < MT1; ++mt) {
                float16_t acc;
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
                for (int s = 0; s < KS1; ++s)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1f[(mt * KS1 + s) * 64], xb[s], acc, 0, 0, 0);
                // acc[i]: hidden channel 32 mt + 8 (i/4) + 4 hl + i%4 of voxel vl
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    const half4_t b4 = *reinterpret_cast<const half4_t*>(bs + 32 * mt + 8 * gq + 4 * hl);
#pragma unroll
                    for (int jj = 0; jj < 4; ++jj) {
                        const half_t hsum = (half_t)((float)(half_t)acc[4 * gq + jj] + (float)b4[jj]);  // fp16 add, RNE
                        hb[2 * mt + gq / 2][4 * (gq % 2) + jj] = hsum > (half_t)0 ? hsum : (half_t)0;
                    }
                }
            }
            load_x(tidx + tiles_per_round);
            // ---- second product ----
#pragma unroll
            for (int mo = 0; mo < MO; ++mo) {
                float16_t acc;
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
                for (int s = 0; s < KS2; ++s)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2f[(mo * KS2 + s) * 64], hb[s], acc, 0, 0, 0);
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    const int co = 32 * mo + 8 * gq + 4 * hl;
                    if (co < C) {
                        half4_t o;
#pragma unroll
                        for (int jj = 0; jj < 4; ++jj) o[jj] = (half_t)acc[4 * gq + jj];
                        *reinterpret_cast<half4_t*>(my + Tile::piece(vl, 4 * mo + gq, hl)) = o;
                    }
                }
            }
            // ---- write-back of the wavefront's own tile: no other wavefront touches it, and the LDS
            // operations of one wavefront complete in issue order, so no workgroup barrier is needed ----
            __builtin_amdgcn_wave_barrier();
            const plane_rsrc_t outr = rows_rsrc(out, tidx * 32, 32, V, 2 * C),
                               addr = rows_rsrc(add, (tidx + tiles_per_round) * 32, 32, V, 2 * C);
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                const int c = k * kWave + lane;
                const int row = c / (C / 8), cc = c % (C / 8);
                half8_t o = Tile::read(my, row, cc);
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) o[jj] = (half_t)((float)o[jj] + (float)ab[k][jj]);  // fp16 add, RNE
                plane_store16<true>(outr, (uint32_t)c * 16, o);
                ab[k] = plane_load16<true>(addr, (uint32_t)c * 16);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// Workgroups per compute unit.  A workgroup begins with its weights, which small volumes notice most (us with 1 / 2 / 3):
// C = 64 at 45000 voxels 10.9 / 12.8 / 13.0, 0.16 M 19.0 / 20.5 / 22.8, 0.2 M 24.1 / 23.5 / 27.1, 2.0 M 161 / 139 / 145;
// C = 32 at 0.1 M 7.9 / 7.4 / 8.6, 0.9 M 39.4 / 31.9 / 33.9, 4.0 M 164 / 133 / 139; C = 16 (2 / 3 / 4) at 0.1 M 4.6 / 5.1
// / 5.1, 0.25 M 7.2 / 6.8 / 7.6, 0.9 M 17.5 / 16.7 / 16.3, 2.0 M 34.7 / 33.6 / 33.5
static int mlp_blocks(int64_t V, int C)
{
    const int64_t per_cu = C == 64 ? (V < 180000 ? 1 : 2) : C == 32 || V < 140000 ? 2 : V < 500000 ? 3 : 4;
    return (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div64(V, 32 * kMlpWaves), per_cu * device_geometry().cus));
}

}  // namespace kerops

using namespace kerops;

extern "C" int kerops_lin_brelu_lin_add_f16(const void* x, const void* Wup, const void* Wdown, const void* bias,
                                            const void* add, void* out, int64_t V, int32_t C, void* stream)
{
    if (!x || !Wup || !Wdown || !bias || !add || !out || !aligned16(x) || !aligned16(add) || !aligned16(out)) {
        set_error("lin_brelu_lin_add: null or misaligned pointer");
        return KEROPS_E_BADARG;
    }
    if (V <= 0) {
        set_error("lin_brelu_lin_add: non-positive size");
        return KEROPS_E_BADARG;
    }
    const int blocks = mlp_blocks(V, C);
    hipStream_t s = (hipStream_t)stream;
#define KEROPS_MLP_CASE(CV)                                                                                        \
    if (C == CV) {                                                                                                 \
        hipLaunchKernelGGL((lin_brelu_lin_add_kernel<CV>), dim3(blocks), dim3(kMlpThreads), 0, s, (const half_t*)x, \
                           (const half_t*)Wup, (const half_t*)Wdown, (const half_t*)bias, (const half_t*)add,       \
                           (half_t*)out, V);                                                                        \
        return check_launch("lin_brelu_lin_add");                                                                  \
    }
    KEROPS_MLP_CASE(16)
    KEROPS_MLP_CASE(32)
    KEROPS_MLP_CASE(64)
#undef KEROPS_MLP_CASE
    set_error("lin_brelu_lin_add: built for C in {16,32,64} (got %d)", C);
    return KEROPS_E_UNSUPPORTED_C;
}

// =============================================================================================
// Backward of the block above, one pass over x and grad:
//
//   linup = fp16(x @ Wup) + bias (fp16 add);  hid = relu(linup)
//   dWdown[h, c] = sum_v hid[v, h] * g[v, c]
//   lg[v, h]     = linup[v, h] > 0 ? fp16(sum_c Wdown[h, c] * g[v, c]) : 0
//   dWup[c, h]   = sum_v x[v, c] * lg[v, h];   dbias[h] = sum_v lg[v, h]
//   dx[v, c]     = fp16(sum_h Wup[c, h] * lg[v, h])
//
// Two kernels: C <= 32 (one block of in / out channels) runs lin_brelu_lin_bwd_wave_kernel further down,
// where a wavefront needs no LDS tiles and no workgroup barrier per tile; C = 64 runs the kernel below.
//
// A workgroup of four wavefronts loops over tiles of 64 voxels; x and g tiles are staged through LDS.
// Phase A: wavefront w computes hidden block w (32 channels) of all 64 voxels, linup^T and (Wdown g^T) with the same
// output layout, applies bias / ReLU / mask in registers and writes the hid and lg tiles to LDS.
// Phase B: dx^T = Wup lg^T from the lg tile (one block of 32 voxels x 32 channels per wavefront, bounced through LDS for
// 16-byte stores), and the reductions over voxels, four 32x32 blocks per wavefront: dWdown = hid^T g (even wavefronts)
// and dWup = x^T lg (odd ones), which stay in fp32 registers for all tiles of the workgroup; their operands, 8 consecutive
// voxels of one channel, are transposing LDS reads (SwizzledRows).  dbias adds up the lg operands that the odd wavefronts
// read anyway.  The weight fragments of phase A are the same for every tile and stay in the wavefront's registers, so that
// the LDS holds two workgroups per compute unit.  Partials go to the workspace, a second kernel adds them in a fixed order
// (fp64): deterministic, no atomics.
// Two workgroups of 256 registers per lane; with operands read from LDS in 2-byte pieces and the weights in LDS, one
// workgroup per compute unit, the op with its reduction took 721 us at 1.96 M voxels, now 247 (its HBM traffic at 6 TB/s:
// 125 us).
namespace kerops {

struct MbCfg {
    static constexpr int C = 64, H = 128, TILE = 64;
    static constexpr int MH = H / 32, MO = C / 32;         // 32-channel blocks of hidden / in-out channels
    static constexpr int KC = C / 16, KH = H / 16;         // k steps over C / over H
    static constexpr int KV = TILE / 16;                   // k steps over the voxels of a tile
    static constexpr int NLX = TILE * C / 8 / kMlpThreads; // 16-byte chunks of an x / g / dx tile per thread
    static constexpr int RW = 2 * C * H + H;               // floats of one partial: dWup, dWdown, dbias
    static constexpr int XS_OFF = 0;
    static constexpr int GS_OFF = XS_OFF + TILE * C * 2;
    static constexpr int HS_OFF = GS_OFF + TILE * C * 2;
    static constexpr int LS_OFF = HS_OFF + TILE * H * 2;
    static constexpr int DS_OFF = LS_OFF + TILE * H * 2;
    static constexpr int A6_OFF = DS_OFF + TILE * C * 2;   // fragments of the dx product [mo][s]
    static constexpr int LDS_BYTES = A6_OFF + MO * KH * 64 * 16;
    static_assert(RW % 32 == 0, "whole lines for the reduction");
    static_assert(MH == kMlpWaves && 2 * MO == kMlpWaves, "one hidden block and one dx block per wavefront");
    static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups per compute unit");
};

__global__ __launch_bounds__(kMlpThreads, 2) void lin_brelu_lin_bwd_kernel(const half_t* __restrict__ x,
                                                                           const half_t* __restrict__ g,
                                                                           const half_t* __restrict__ Wup,
                                                                           const half_t* __restrict__ Wdown,
                                                                           const half_t* __restrict__ bias,
                                                                           half_t* __restrict__ dx,
                                                                           float* __restrict__ ws, int64_t V)
{
    using Cfg = MbCfg;
    constexpr int C = Cfg::C, H = Cfg::H, KC = Cfg::KC, KH = Cfg::KH, KV = Cfg::KV, NLX = Cfg::NLX, TILE = Cfg::TILE;
    using XT = SwizzledRows<C>;  // x and g tiles
    using HT = SwizzledRows<H>;  // hid and lg tiles
    __shared__ __attribute__((aligned(16))) unsigned char smem[Cfg::LDS_BYTES];
    unsigned char* xs = smem + Cfg::XS_OFF;
    unsigned char* gs = smem + Cfg::GS_OFF;
    unsigned char* hs = smem + Cfg::HS_OFF;
    unsigned char* ls = smem + Cfg::LS_OFF;
    unsigned char* ds = smem + Cfg::DS_OFF;

    const int t = threadIdx.x, lane = t % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
    const int il = lane % 32, hl = lane / 32;
    const half8_t z8 = {0, 0, 0, 0, 0, 0, 0, 0};

    // fragments of the three per-voxel products (lane: row il of the block, k = 16 s + 8 hl + 0..7)
    half8_t a1[KC], a3[KC];
    half4_t b4[4];
    const int mo = wave / 2, vto = wave % 2;  // the wavefront's dx block
#pragma unroll
    for (int s = 0; s < KC; ++s) {
#pragma unroll
        for (int j = 0; j < 8; ++j) a1[s][j] = Wup[(16 * s + 8 * hl + j) * H + 32 * wave + il];  // linup^T = Wup^T x^T
        a3[s] = load_c8(Wdown + (32 * wave + il) * C + 16 * s + 8 * hl);                        // Wdown g^T
    }
    half8_t* a6w = reinterpret_cast<half8_t*>(smem + Cfg::A6_OFF);  // dx^T = Wup lg^T
    constexpr int N6 = Cfg::MO * KH * 64 / kMlpThreads;
    half8_t w6[N6];
#pragma unroll
    for (int k = 0; k < N6; ++k) {
        const int i = t + k * kMlpThreads, l = i % 64, s = (i / 64) % KH, m = i / (64 * KH);
        w6[k] = load_c8(Wup + (32 * m + l % 32) * H + 16 * s + 8 * (l / 32));
    }
#pragma unroll
    for (int k = 0; k < N6; ++k) a6w[t + k * kMlpThreads] = w6[k];
    const half8_t* a6 = a6w + mo * KH * 64 + lane;  // (the barrier behind the first staging covers it)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) b4[gq][jj] = bias[32 * wave + 8 * gq + 4 * hl + jj];

    // reduction blocks of this wavefront, k = 0..3: hidden block mh = wave / 2 + 2 (k % 2), in-out block mc = k / 2;
    // even wavefronts: dWdown[h, c] = hid^T g, odd ones: dWup[c, h] = x^T lg
    float16_t wacc[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < 16; ++i) wacc[k][i] = 0.0f;
    float bacc[2] = {0.0f, 0.0f};  // odd wavefronts: dbias of hidden block wave / 2 + 2 k, channel il
    int hoff[2][2], xoff[2][2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        HT::tr_offsets(lane, wave / 2 + 2 * k, hoff[k]);
        XT::tr_offsets(lane, k, xoff[k]);
    }

    const int64_t ntiles = (V + TILE - 1) / TILE;
    // (nothing behind a condition, see rows_rsrc: a tile waits for its loads and leaves the stores of the one before in
    // flight: 273 -> 247 us at 2.0 M voxels)
    half8_t xpre[NLX], gpre[NLX];
    auto prefetch = [&](int64_t tile) {
        const plane_rsrc_t xr = rows_rsrc(x, tile * TILE, TILE, V, 2 * C), gr = rows_rsrc(g, tile * TILE, TILE, V, 2 * C);
#pragma unroll
        for (int j = 0; j < NLX; ++j) {
            xpre[j] = plane_load16<true>(xr, (uint32_t)(t + j * kMlpThreads) * 16);
            gpre[j] = plane_load16<true>(gr, (uint32_t)(t + j * kMlpThreads) * 16);
        }
    };

    int64_t tile = blockIdx.x;
    prefetch(tile);
#pragma unroll
    for (int j = 0; j < NLX; ++j) plane_store16<true>(plane_rsrc(dx, 0u), 0u, z8);  // (of nothing: as many as a tile's)
    for (; tile < ntiles; tile += gridDim.x) {
        // ---- stage the tile (rows past V are zero: they add nothing to the reductions) ----
        // (the previous tile's x and g were last read before the barrier in front of its write-back)
#pragma unroll
        for (int j = 0; j < NLX; ++j) {
            const int c = t + j * kMlpThreads;
            const int off = XT::chunk16(c / (C / 8), c % (C / 8));
            *reinterpret_cast<half8_t*>(xs + off) = xpre[j];
            *reinterpret_cast<half8_t*>(gs + off) = gpre[j];
        }
        __syncthreads();
        prefetch(tile + gridDim.x);

        // ---- phase A: hid and lg, 32 voxels x 32 hidden channels at a time ----
#pragma unroll 1  // (unrolled, the offsets of both halves cost spilled registers)
        for (int vt = 0; vt < 2; ++vt) {
            const int row = 32 * vt + il;
            // chunk 2 s + hl of the row: the swizzle is an XOR, so step s is the offset of step 0 ^ 32 s
            const int xrow = XT::chunk16(row, hl);
            float16_t up, dn;
#pragma unroll
            for (int i = 0; i < 16; ++i) up[i] = dn[i] = 0.0f;
#pragma unroll
            for (int s = 0; s < KC; ++s) {
                const half8_t xb = *reinterpret_cast<const half8_t*>(xs + (xrow ^ (32 * s)));
                const half8_t gb = *reinterpret_cast<const half8_t*>(gs + (xrow ^ (32 * s)));
                up = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1[s], xb, up, 0, 0, 0);
                dn = __builtin_amdgcn_mfma_f32_32x32x16_f16(a3[s], gb, dn, 0, 0, 0);
            }
            // up[i], dn[i]: hidden channel 32 wave + 8 (i/4) + 4 hl + i%4 of voxel row
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                half4_t hv, lv;
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const half_t lin = (half_t)((float)(half_t)up[4 * gq + jj] + (float)b4[gq][jj]);  // fp16 add
                    const bool pos = lin > (half_t)0;
                    hv[jj] = pos ? lin : (half_t)0;
                    lv[jj] = pos ? (half_t)dn[4 * gq + jj] : (half_t)0;
                }
                // rows past V hold x = g = 0: hid = relu(bias) there, which must not reach dWdown ... but
                // it is multiplied by g = 0; lg = fp16(0) = 0, so dWup and dbias are unaffected as well
                const int off = HT::chunk16(row, 4 * wave + gq) + 8 * hl;
                *reinterpret_cast<half4_t*>(hs + off) = hv;
                *reinterpret_cast<half4_t*>(ls + off) = lv;
            }
        }
        __syncthreads();

        // ---- phase B1: the dx^T block (vto, mo) from the lg tile ----
        {
            const int row = 32 * vto + il;
            const int lrow = HT::chunk16(row, hl);
            float16_t acc;
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
            for (int s = 0; s < KH; ++s) {
                const half8_t lb = *reinterpret_cast<const half8_t*>(ls + (lrow ^ (32 * s)));
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a6[64 * s], lb, acc, 0, 0, 0);
            }
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                half4_t o;
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) o[jj] = (half_t)acc[4 * gq + jj];
                *reinterpret_cast<half4_t*>(ds + BounceTile<C>::piece(row, 4 * mo + gq, hl)) = o;
            }
        }
        // ---- phase B2: the reductions over the voxels of the tile ----
#pragma unroll
        for (int s = 0; s < KV; ++s) {
            if (wave % 2 == 0) {
                const half8_t hf[2] = {HT::read_tr(hs, hoff[0], s), HT::read_tr(hs, hoff[1], s)};
                const half8_t gf[2] = {XT::read_tr(gs, xoff[0], s), XT::read_tr(gs, xoff[1], s)};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    wacc[k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hf[k % 2], gf[k / 2], wacc[k], 0, 0, 0);
            } else {
                const half8_t lf[2] = {HT::read_tr(ls, hoff[0], s), HT::read_tr(ls, hoff[1], s)};
                const half8_t xf[2] = {XT::read_tr(xs, xoff[0], s), XT::read_tr(xs, xoff[1], s)};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    wacc[k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[k / 2], lf[k % 2], wacc[k], 0, 0, 0);
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int j = 0; j < 8; ++j) bacc[k] += (float)lf[k][j];
            }
        }
        __syncthreads();

        // ---- phase C: dx write-back, 16-byte chunks (the dx tile is written next behind two barriers) ----
        const plane_rsrc_t dr = rows_rsrc(dx, tile * TILE, TILE, V, 2 * C);
#pragma unroll
        for (int j = 0; j < NLX; ++j) {
            const int c = t + j * kMlpThreads;
            const int row = c / (C / 8), cc = c % (C / 8);
            plane_store16<true>(dr, (uint32_t)c * 16, BounceTile<C>::read(ds, row, cc));
        }
    }

    // ---- partials of this workgroup: row blockIdx = [dWup C*H][dWdown H*C][dbias H] ----
    float* out = ws + (int64_t)blockIdx.x * Cfg::RW;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int mh = wave / 2 + 2 * (k % 2), mc = k / 2;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int ri = 8 * (i / 4) + 4 * hl + i % 4;  // row of the block held in register i
            if (wave % 2 == 0) out[C * H + (32 * mh + ri) * C + 32 * mc + il] = wacc[k][i];  // D[h][c]
            else out[(32 * mc + ri) * H + 32 * mh + il] = wacc[k][i];                        // D[c][h]
        }
    }
    if (wave % 2 == 1) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float sum = bacc[k] + __shfl_xor(bacc[k], 32, 64);  // the two lane halves hold different voxels
            if (hl == 0) out[2 * C * H + 32 * (wave / 2 + 2 * k) + il] = sum;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// C <= 32: every wavefront works alone on tiles of 32 voxels, no workgroup barrier inside the loop.
//
// The per-voxel products want "voxel per lane" results (lane = voxel, registers = channels: the B operand
// of the next per-voxel product), the reductions over voxels want "channel per lane" operands (lane =
// channel, registers = 8 voxels).  A 32x32 matrix-core block D = A B holds column j in lane j%32, so the
// second form of a tile M[v][c] is the product M I with an identity B fragment: exact, since every sum has
// one non-zero term.  Fragments of x and g come straight from global memory (16-byte chunk 2 s + l/32 of
// voxel l%32: the same registers serve as A operand of the transposing product and B operand of the
// per-voxel products); hid and lg are transposed from their packed fp16 registers, whose reduction index
// runs over the hidden channels in the order the accumulator leaves them, with a matching permuted
// identity.  Weight and identity fragments sit in LDS (one 16-byte read per lane and use).  The
// accumulators of dWup, dWdown and dbias stay in registers for all tiles of the wavefront; at the end the
// four wavefronts add theirs in LDS in a fixed order and the workgroup writes one partial row.
template <int C>
struct MtCfg {
    static constexpr int H = 2 * C;
    static constexpr int MH = H / 32;   // 32-channel blocks of the hidden channels
    static constexpr int KC = C / 16;   // k steps over the in / out channels
    static constexpr int DP = C;        // row pitch of the dx tile (halves): dense rows, BounceTile in common.hpp
    static constexpr int RW = 2 * C * H + H;
    static constexpr int F1_OFF = 0;                              // Wup^T rows   [mh][s]
    static constexpr int F2_OFF = F1_OFF + MH * KC * 1024;        // Wdown rows   [mh][s]
    static constexpr int F3_OFF = F2_OFF + MH * KC * 1024;        // Wup rows, hidden order of the accumulator
    static constexpr int IP_OFF = F3_OFF + 2 * MH * 1024;         // identity in that order [half]
    static constexpr int ID_OFF = IP_OFF + 2 * 1024;              // identity [s]
    static constexpr int BH_OFF = ID_OFF + KC * 1024;             // bias
    static constexpr int DS_OFF = (BH_OFF + H * 2 + 15) / 16 * 16;
    static constexpr int LOOP_BYTES = DS_OFF + kMlpWaves * 32 * DP * 2;
    static constexpr int LDS_BYTES = LOOP_BYTES > RW * 4 ? LOOP_BYTES : RW * 4;
    static_assert(C == 16 || C == 32, "one 32-channel block of in / out channels");
    static_assert(RW % 32 == 0, "whole lines for the reduction");
};

// fp32 accumulator -> the two packed fp16 operands (registers 0..7 and 8..15)
__device__ __forceinline__ void pack_acc(const float16_t& a, half8_t& lo, half8_t& hi)
{
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        lo[i] = (half_t)a[i];
        hi[i] = (half_t)a[8 + i];
    }
}

typedef short i16x2_t __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

// Two neighbouring accumulator registers of both products -> packed (hid, lg), 16-bit packed operations only:
// lin = fp16(up) + bias (fp16 add);  hid = relu(lin) as the signed integer maximum of the bit pattern with 0
// (negative values and -0 have the sign bit set, positive ones compare like integers);  lg = fp16(dn) where
// hid has a non-zero bit pattern, i.e. where lin > 0.
__device__ __forceinline__ void hid_lg_pair(float u0, float u1, float d0, float d1, half2_t b, half2_t& hid,
                                            half2_t& lg)
{
    const half2_t up2 = {(half_t)u0, (half_t)u1};
    const half2_t dn2 = {(half_t)d0, (half_t)d1};
    const half2_t lin = up2 + b;
    const i16x2_t hb = __builtin_elementwise_max(__builtin_bit_cast(i16x2_t, lin), i16x2_t{0, 0});
    hid = __builtin_bit_cast(half2_t, hb);
    const u16x2_t one = {1, 1}, zero = {0, 0};
    uint32_t nz;  // written out: the compiler would turn the minimum into two compares and selects
    asm("v_pk_min_u16 %0, %1, %2" : "=v"(nz) : "v"(__builtin_bit_cast(uint32_t, hb)), "v"(__builtin_bit_cast(uint32_t, one)));
    const u16x2_t m = zero - __builtin_bit_cast(u16x2_t, nz);  // 0 or 0xffff per half
    lg = __builtin_bit_cast(half2_t, __builtin_bit_cast(uint32_t, dn2) & __builtin_bit_cast(uint32_t, m));
}

template <int C>
__global__ __launch_bounds__(kMlpThreads, 2) void lin_brelu_lin_bwd_wave_kernel(
    const half_t* __restrict__ x, const half_t* __restrict__ g, const half_t* __restrict__ Wup,
    const half_t* __restrict__ Wdown, const half_t* __restrict__ bias, half_t* __restrict__ dx,
    float* __restrict__ ws, int64_t V)
{
    using Cfg = MtCfg<C>;
    constexpr int H = Cfg::H, MH = Cfg::MH, KC = Cfg::KC, DP = Cfg::DP;
    __shared__ __attribute__((aligned(16))) unsigned char smem[Cfg::LDS_BYTES];
    half_t* f1w = reinterpret_cast<half_t*>(smem + Cfg::F1_OFF);
    half_t* f3w = reinterpret_cast<half_t*>(smem + Cfg::F3_OFF);
    half_t* ipw = reinterpret_cast<half_t*>(smem + Cfg::IP_OFF);
    half_t* idw = reinterpret_cast<half_t*>(smem + Cfg::ID_OFF);
    half_t* bsh = reinterpret_cast<half_t*>(smem + Cfg::BH_OFF);

    const int t = threadIdx.x, lane = t % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(t / kWave);  // scalar: tile indices stay wavefront-uniform
    const int il = lane % 32, hl = lane / 32;
    const half8_t z8 = {0, 0, 0, 0, 0, 0, 0, 0};

    // hidden channel (within a block of 32) that element j of reduction group `half` of lane half hl holds
    auto hperm = [](int half, int hl_, int j) { return 16 * half + 8 * (j / 4) + 4 * hl_ + j % 4; };

    for (int i = t; i < MH * KC * 512; i += kMlpThreads) {
        const int j = i % 8, l = (i / 8) % 64, s = (i / 512) % KC, mh = i / (512 * KC);
        f1w[i] = Wup[(16 * s + 8 * (l / 32) + j) * H + 32 * mh + l % 32];
    }
    for (int i = t; i < MH * KC * 64; i += kMlpThreads) {
        const int l = i % 64, s = (i / 64) % KC, mh = i / (64 * KC);
        reinterpret_cast<half8_t*>(smem + Cfg::F2_OFF)[i] = load_c8(Wdown + (32 * mh + l % 32) * C + 16 * s + 8 * (l / 32));
    }
    for (int i = t; i < 2 * MH * 512; i += kMlpThreads) {
        const int j = i % 8, l = (i / 8) % 64, f = i / 512;
        const int c = l % 32, h = 32 * (f / 2) + hperm(f % 2, l / 32, j);
        f3w[i] = c < C ? Wup[c * H + h] : (half_t)0;
    }
    for (int i = t; i < 2 * 512; i += kMlpThreads) {
        const int j = i % 8, l = (i / 8) % 64, half = i / 512;
        ipw[i] = hperm(half, l / 32, j) == l % 32 ? (half_t)1 : (half_t)0;
    }
    for (int i = t; i < KC * 512; i += kMlpThreads) {
        const int j = i % 8, l = (i / 8) % 64, s = i / 512;
        idw[i] = 16 * s + 8 * (l / 32) + j == l % 32 ? (half_t)1 : (half_t)0;
    }
    for (int i = t; i < H; i += kMlpThreads) bsh[i] = bias[i];
    __syncthreads();

    const half8_t* f1 = reinterpret_cast<const half8_t*>(smem + Cfg::F1_OFF) + lane;
    const half8_t* f2 = reinterpret_cast<const half8_t*>(smem + Cfg::F2_OFF) + lane;
    const half8_t* f3 = reinterpret_cast<const half8_t*>(smem + Cfg::F3_OFF) + lane;
    const half8_t* ip = reinterpret_cast<const half8_t*>(smem + Cfg::IP_OFF) + lane;
    const half8_t* id = reinterpret_cast<const half8_t*>(smem + Cfg::ID_OFF) + lane;
    unsigned char* my = smem + Cfg::DS_OFF + wave * 32 * DP * 2;
    using Tile = BounceTile<C>;

    float16_t wdn[MH], wup[MH];  // dWdown block: D[h][c];  dWup block: D[c][h]
    float bacc[MH];
#pragma unroll
    for (int mh = 0; mh < MH; ++mh) {
#pragma unroll
        for (int i = 0; i < 16; ++i) wdn[mh][i] = wup[mh][i] = 0.0f;
        bacc[mh] = 0.0f;
    }

    const int64_t ntiles = (V + 31) / 32;
    const int64_t stride = (int64_t)gridDim.x * kMlpWaves;
    half8_t xn[KC], gn[KC];
    auto fetch = [&](int64_t tile) {  // rows past V read the last voxel and are zeroed before use
        int64_t v = tile * 32 + il;
        v = v < V ? v : V - 1;
#pragma unroll
        for (int s = 0; s < KC; ++s) {
            xn[s] = load_c8_nt(x + v * C + 16 * s + 8 * hl);
            gn[s] = load_c8_nt(g + v * C + 16 * s + 8 * hl);
        }
    };

    // dx leaves one tile late: the wait for the operands of a tile then only covers stores issued a whole
    // tile earlier (the memory counter retires loads and stores in issue order)
    auto flush = [&](int64_t pv0, bool ragged) {
#pragma unroll
        for (int c0 = 0; c0 < 32 * C / 8; c0 += kWave) {
            const int c = c0 + lane;
            const int row = c / (C / 8), cc = c % (C / 8);
            if (!ragged || pv0 + row < V) {
                store_c8_nt(dx + (pv0 + row) * C + cc * 8, Tile::read(my, row, cc));
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    const int64_t first = (int64_t)blockIdx.x * kMlpWaves + wave;
    int64_t tile = first;
    if (tile < ntiles) fetch(tile);
    for (; tile < ntiles; tile += stride) {
        const int64_t v0 = tile * 32;
        half8_t xc[KC], gc[KC];
#pragma unroll
        for (int s = 0; s < KC; ++s) {
            xc[s] = xn[s];
            gc[s] = gn[s];
        }
        if (v0 + 32 > V) {  // ragged last tile (wavefront-uniform)
            const bool ok = v0 + il < V;
#pragma unroll
            for (int s = 0; s < KC; ++s) {
                xc[s] = ok ? xc[s] : z8;
                gc[s] = ok ? gc[s] : z8;
            }
        }
        if (tile != first) flush(v0 - stride * 32, false);  // an earlier tile of this wavefront is never ragged
        {
            const int64_t nt = tile + stride;
            fetch(nt < ntiles ? nt : tile);
        }
        __builtin_amdgcn_sched_barrier(0);

        // x^T, g^T: lane = channel, registers = voxels 8 (i/4) + 4 hl + i%4
        half8_t xT[2], gT[2];
        {
            float16_t tx, tg;
#pragma unroll
            for (int i = 0; i < 16; ++i) tx[i] = tg[i] = 0.0f;
#pragma unroll
            for (int s = 0; s < KC; ++s) {
                const half8_t e = id[s * 64];
                tx = __builtin_amdgcn_mfma_f32_32x32x16_f16(xc[s], e, tx, 0, 0, 0);
                tg = __builtin_amdgcn_mfma_f32_32x32x16_f16(gc[s], e, tg, 0, 0, 0);
            }
            pack_acc(tx, xT[0], xT[1]);
            pack_acc(tg, gT[0], gT[1]);
        }

        float16_t dacc;  // dx^T: D[c][v]
#pragma unroll
        for (int i = 0; i < 16; ++i) dacc[i] = 0.0f;

#pragma unroll
        for (int mh = 0; mh < MH; ++mh) {
            float16_t up, dn;
#pragma unroll
            for (int i = 0; i < 16; ++i) up[i] = dn[i] = 0.0f;
#pragma unroll
            for (int s = 0; s < KC; ++s) {
                up = __builtin_amdgcn_mfma_f32_32x32x16_f16(f1[(mh * KC + s) * 64], xc[s], up, 0, 0, 0);
                dn = __builtin_amdgcn_mfma_f32_32x32x16_f16(f2[(mh * KC + s) * 64], gc[s], dn, 0, 0, 0);
            }
            // up[i], dn[i]: hidden channel 32 mh + 8 (i/4) + 4 hl + i%4 of voxel il
            half8_t hv[2], lv[2];
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                const half4_t b4 = *reinterpret_cast<const half4_t*>(bsh + 32 * mh + 8 * gq + 4 * hl);
#pragma unroll
                for (int jp = 0; jp < 2; ++jp) {
                    const int i = 4 * gq + 2 * jp, e = 4 * (gq % 2) + 2 * jp;
                    half2_t hid, lg;
                    hid_lg_pair(up[i], up[i + 1], dn[i], dn[i + 1], half2_t{b4[2 * jp], b4[2 * jp + 1]}, hid, lg);
                    hv[gq / 2][e] = hid[0];
                    hv[gq / 2][e + 1] = hid[1];
                    lv[gq / 2][e] = lg[0];
                    lv[gq / 2][e + 1] = lg[1];
                }
            }
            // rows past V hold x = g = 0: hid = relu(bias) there meets g = 0 in dWdown, lg = 0 everywhere else
            dacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f3[(2 * mh) * 64], lv[0], dacc, 0, 0, 0);
            dacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f3[(2 * mh + 1) * 64], lv[1], dacc, 0, 0, 0);

            // hid^T, lg^T: lane = hidden channel 32 mh + il, registers = voxels
            half8_t hT[2], lT[2];
            {
                float16_t th, tl;
#pragma unroll
                for (int i = 0; i < 16; ++i) th[i] = tl[i] = 0.0f;
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    const half8_t e = ip[hf * 64];
                    th = __builtin_amdgcn_mfma_f32_32x32x16_f16(hv[hf], e, th, 0, 0, 0);
                    tl = __builtin_amdgcn_mfma_f32_32x32x16_f16(lv[hf], e, tl, 0, 0, 0);
                }
                pack_acc(th, hT[0], hT[1]);
#pragma unroll
                for (int i = 0; i < 16; ++i) bacc[mh] += tl[i];
                pack_acc(tl, lT[0], lT[1]);
            }
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                wdn[mh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hT[hf], gT[hf], wdn[mh], 0, 0, 0);
                wup[mh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xT[hf], lT[hf], wup[mh], 0, 0, 0);
            }
        }

        // ---- dx: into the wavefront's own LDS tile; the LDS operations of one wavefront complete in issue
        // order, so no workgroup barrier is needed ----
#pragma unroll
        for (int gq = 0; gq < C / 8; ++gq) {
            half4_t o;
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) o[jj] = (half_t)dacc[4 * gq + jj];
            *reinterpret_cast<half4_t*>(my + Tile::piece(il, gq, hl)) = o;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (first < ntiles) flush((tile - stride) * 32, true);

    // ---- the four wavefronts add their partials in LDS, wavefront 0 first: [dWup C*H][dWdown H*C][dbias H] ----
    float* red = reinterpret_cast<float*>(smem);
    __syncthreads();  // every wavefront is done with the fragments
#pragma unroll 1
    for (int w = 0; w < kMlpWaves; ++w) {
        if (wave == w) {
#pragma unroll
            for (int mh = 0; mh < MH; ++mh) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int ri = 8 * (i / 4) + 4 * hl + i % 4;  // row of the block held in register i
                    if (il < C) {  // dWdown[h = 32 mh + ri][c = il]
                        float* p = red + C * H + (32 * mh + ri) * C + il;
                        *p = w == 0 ? wdn[mh][i] : *p + wdn[mh][i];
                    }
                    if (ri < C) {  // dWup[c = ri][h = 32 mh + il]
                        float* p = red + ri * H + 32 * mh + il;
                        *p = w == 0 ? wup[mh][i] : *p + wup[mh][i];
                    }
                }
                const float b = bacc[mh] + __shfl_xor(bacc[mh], 32);  // both lane halves hold 16 voxels each
                if (hl == 0) {
                    float* p = red + 2 * C * H + 32 * mh + il;
                    *p = w == 0 ? b : *p + b;
                }
            }
        }
        __syncthreads();
    }
    float* out = ws + (int64_t)blockIdx.x * Cfg::RW;
    for (int i = t; i < Cfg::RW; i += kMlpThreads) out[i] = red[i];
}

// ---------------------------------------------------------------------------------------------
// C = 32 with transposing LDS reads.
//
// Same tiles, products and accumulators as lin_brelu_lin_bwd_wave_kernel; what differs is how the "channel per
// lane" operands of the two weight-gradient products are made.  gfx950 reads LDS transposed: ds_read_b64_tr_b16
// takes, in every block of 16 lanes, the 16 x 4 matrix M of 16-bit values that the lanes address (lane s supplies
// the address of four consecutive values M[s][0..3]) and returns to lane i the values M[4 j + i/4][i%4], j = 0..3.
// With lane s pointing at row s/4, columns 4 (s%4) .. 4 (s%4) + 3 of a row-major [voxel][channel] tile, lane i
// receives channel i of four consecutive voxels: one instruction transposes a 4 x 16 patch, two of them make the
// eight reduction values of a 32x32x16 operand.  So the x, g, hid and lg tiles of a wavefront are written to its own
// LDS area as they sit in the registers (one 64-byte row per voxel) and read back transposed, instead of being
// multiplied with an identity on the matrix cores and converted back to fp16: 12 of 32 matrix instructions and the
// conversions of their results go.
// LDS layout: measured on gfx950, reads see 64 banks of 4 bytes (32 lanes of an 8-byte read or 16 lanes of a 16-byte
// read per clock), writes see 32 (16 lanes of an 8-byte write, 8 lanes of a 16-byte write per clock).  Chunk c of
// row r sits in chunk slot c ^ tr_slot(r) = c ^ ((r / 2) % 4) ^ ((r / 8) % 2): the eight rows of a write phase then
// cover the 128 bytes of write banks once, the sixteen rows of a 16-byte read phase (the same chunk of each) the 256
// of read banks once, and a transposing read phase takes four whole rows.
// x and g are fetched as whole rows (one instruction = 16 voxels x 64 bytes = 1 KB of consecutive memory) into the
// tiles; the lane's own row comes back from there as the operand of the per-voxel products.
// The hidden channels of a tile row are stored in the order the accumulator leaves them (position p of the row is
// hidden channel tr_hidden(p) of the 32-block), which only permutes the rows / columns of the gradient blocks.
// The bias gradient is a product of its own on the 16x16x32 instruction: an operand of ones in row 0 for the even
// 16-lane groups and in row 1 for the odd ones adds the lg values of hidden positions 0..15 and 16..31.
struct MrCfg {
    static constexpr int C = 32, H = 64, MH = 2, KC = 2;
    static constexpr int RW = 2 * C * H + H;
    static constexpr int F1_OFF = 0;                              // Wup^T rows   [mh][s]
    static constexpr int F2_OFF = F1_OFF + MH * KC * 1024;        // Wdown rows   [mh][s]
    static constexpr int F3_OFF = F2_OFF + MH * KC * 1024;        // Wup rows, hidden order of the accumulator
    static constexpr int BH_OFF = F3_OFF + 2 * MH * 1024;         // bias
    static constexpr int WV_OFF = (BH_OFF + H * 2 + 15) / 16 * 16;
    static constexpr int TILE = 32 * 64;                          // one [32 voxels][32 values] fp16 tile
    static constexpr int WV_BYTES = 5 * TILE;                     // per wavefront: x, g, hid, lg, dx
    static constexpr int LOOP_BYTES = WV_OFF + kMlpWaves * WV_BYTES;
    static constexpr int LDS_BYTES = LOOP_BYTES > RW * 4 ? LOOP_BYTES : RW * 4;
};

// chunk-slot swizzle of tile row r (unchanged by r + 16)
__host__ __device__ constexpr int tr_slot(int r) { return ((r >> 1) & 3) ^ ((r >> 3) & 1); }
// hidden channel (inside its block of 32) stored at position p of a tile row
__host__ __device__ constexpr int tr_hidden(int p) { return 16 * (p / 16) + 8 * ((p % 8) / 4) + 4 * ((p / 8) % 2) + p % 4; }


__global__ __launch_bounds__(kMlpThreads, 2) void lin_brelu_lin_bwd_tr_kernel(
    const half_t* __restrict__ x, const half_t* __restrict__ g, const half_t* __restrict__ Wup,
    const half_t* __restrict__ Wdown, const half_t* __restrict__ bias, half_t* __restrict__ dx,
    float* __restrict__ ws, int64_t V)
{
    using Cfg = MrCfg;
    constexpr int C = Cfg::C, H = Cfg::H, MH = Cfg::MH, KC = Cfg::KC, TILE = Cfg::TILE;
    __shared__ __attribute__((aligned(16))) unsigned char smem[Cfg::LDS_BYTES];
    half_t* f1w = reinterpret_cast<half_t*>(smem + Cfg::F1_OFF);
    half_t* f3w = reinterpret_cast<half_t*>(smem + Cfg::F3_OFF);
    half_t* bsh = reinterpret_cast<half_t*>(smem + Cfg::BH_OFF);

    const int t = threadIdx.x, lane = t % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(t / kWave);  // scalar: tile indices stay wavefront-uniform
    const int il = lane % 32, hl = lane / 32;

    // hidden channel (within a block of 32) that element j of reduction group `half` of lane half hl holds
    auto hperm = [](int half, int hl_, int j) { return 16 * half + 8 * (j / 4) + 4 * hl_ + j % 4; };

    // (all loads in flight at once)
    {
        constexpr int N1 = MH * KC * 512 / kMlpThreads, N3 = 2 * MH * 512 / kMlpThreads;
        static_assert(MH * KC * 64 == kMlpThreads && H <= kMlpThreads, "one chunk of Wdown, at most one bias value per thread");
        half_t w1[N1], w3[N3];
#pragma unroll
        for (int k = 0; k < N1; ++k) {
            const int i = t + k * kMlpThreads, j = i % 8, l = (i / 8) % 64, s = (i / 512) % KC, mh = i / (512 * KC);
            w1[k] = Wup[(16 * s + 8 * (l / 32) + j) * H + 32 * mh + l % 32];
        }
#pragma unroll
        for (int k = 0; k < N3; ++k) {
            const int i = t + k * kMlpThreads, j = i % 8, l = (i / 8) % 64, f = i / 512;
            w3[k] = Wup[(l % 32) * H + 32 * (f / 2) + hperm(f % 2, l / 32, j)];
        }
        const int l2 = t % 64, s2 = (t / 64) % KC, mh2 = t / (64 * KC);
        const half8_t w2 = load_c8(Wdown + (32 * mh2 + l2 % 32) * C + 16 * s2 + 8 * (l2 / 32));
        const half_t bias_t = bias[t % H];
#pragma unroll
        for (int k = 0; k < N1; ++k) f1w[t + k * kMlpThreads] = w1[k];
#pragma unroll
        for (int k = 0; k < N3; ++k) f3w[t + k * kMlpThreads] = w3[k];
        reinterpret_cast<half8_t*>(smem + Cfg::F2_OFF)[t] = w2;
        if (t < H) bsh[t] = bias_t;
    }
    __syncthreads();

    const half8_t* f1 = reinterpret_cast<const half8_t*>(smem + Cfg::F1_OFF) + lane;
    const half8_t* f2 = reinterpret_cast<const half8_t*>(smem + Cfg::F2_OFF) + lane;
    const half8_t* f3 = reinterpret_cast<const half8_t*>(smem + Cfg::F3_OFF) + lane;
    unsigned char* mine = smem + Cfg::WV_OFF + wave * Cfg::WV_BYTES;
    unsigned char* xt = mine;             // [32 voxels][32 channels]
    unsigned char* gt = mine + TILE;
    unsigned char* ht = mine + 2 * TILE;  // [32 voxels][32 hidden positions] of the current block
    unsigned char* lt = mine + 3 * TILE;
    unsigned char* dt = mine + 4 * TILE;  // [32 voxels][32 channels] of dx

    // the lane's row: 16-byte chunks hl and 2 + hl
    const int wsw = tr_slot(il);
    const int woff0 = il * 64 + ((hl ^ wsw) * 16), woff1 = il * 64 + (((2 + hl) ^ wsw) * 16);
    // the fetched chunk: row lane / 4 (+ 16 for the second instruction: the same swizzle term), chunk lane % 4
    const int foff = (lane / 4) * 64 + (((lane % 4) ^ tr_slot(lane / 4)) * 16);
    // transposing read of reduction half hf: lane (il, hl) receives position il of the voxels 16 hf + 8 hl + 0..7;
    // inside its block of 16 lanes, lane s addresses row 8 hl + 4 r + s/4, positions 16 (block % 2) + 4 (s%4) ..
    // (rows 16 hf + ...: the swizzle term does not depend on hf)
    int toff[2];
    {
        const int s = lane % 16, blk = lane / 16;
        const int pos = 16 * (blk % 2) + 4 * (s % 4);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int row = 8 * (blk / 2) + 4 * r + s / 4;
            toff[r] = row * 64 + (((pos / 8) ^ tr_slot(row)) * 16) + (pos % 8) * 2;
        }
    }
    auto read_T = [&](const unsigned char* tile, int hf) {
        const half4_t a = lds_read_tr16(tile + hf * 1024 + toff[0]);
        const half4_t b = lds_read_tr16(tile + hf * 1024 + toff[1]);
        return half8_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    };
    auto wave_sync = [] {  // LDS operations of one wavefront complete in issue order: only the compiler must not reorder
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // bias gradient: ones in row 0 for the even 16-lane groups, in row 1 for the odd ones
    const half_t one_h = (lane % 16) == ((lane / 16) % 2) ? (half_t)1 : (half_t)0;
    const half8_t ones = {one_h, one_h, one_h, one_h, one_h, one_h, one_h, one_h};

    float16_t wdn[MH], wup[MH];  // dWdown block: D[h][c];  dWup block: D[c][h]
    float4_t bacc[MH];
#pragma unroll
    for (int mh = 0; mh < MH; ++mh) {
#pragma unroll
        for (int i = 0; i < 16; ++i) wdn[mh][i] = wup[mh][i] = 0.0f;
        bacc[mh] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }

    const int64_t ntiles = (V + 31) / 32;
    const int64_t stride = (int64_t)gridDim.x * kMlpWaves;
    half8_t xn[KC], gn[KC];
    // one instruction fetches 16 whole rows (1 KB): lane -> 16-byte chunk lane % 4 of voxel 16 s + lane / 4
    // (rows that do not exist: zeros)
    auto fetch = [&](int64_t tile) {
        const plane_rsrc_t xr = rows_rsrc(x, tile * 32, 32, V, 2 * C), gr = rows_rsrc(g, tile * 32, 32, V, 2 * C);
#pragma unroll
        for (int s = 0; s < KC; ++s) {
            xn[s] = plane_load16<true>(xr, (uint32_t)(s * kWave + lane) * 16);
            gn[s] = plane_load16<true>(gr, (uint32_t)(s * kWave + lane) * 16);
        }
    };

    // dx leaves one tile late, behind the loads of the tile after it: the wait for the operands of a tile leaves the
    // stores in flight (nothing stands behind a condition, see rows_rsrc)
    auto flush = [&](int64_t pv0) {
        const plane_rsrc_t dr = rows_rsrc(dx, pv0, 32, V, 2 * C);
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {  // lane -> 16-byte chunk lane % 4 of row 16 pass + lane / 4
            const int row = 16 * pass + lane / 4, cc = lane % 4;
            const half8_t o = *reinterpret_cast<const half8_t*>(dt + row * 64 + ((cc ^ tr_slot(row)) * 16));
            // rows 8..15 and 24..31 hold the two 8-byte halves of a chunk swapped
            const bool sw = (row >> 3) & 1;
            const half8_t w = {sw ? o[4] : o[0], sw ? o[5] : o[1], sw ? o[6] : o[2], sw ? o[7] : o[3],
                               sw ? o[0] : o[4], sw ? o[1] : o[5], sw ? o[2] : o[6], sw ? o[3] : o[7]};
            plane_store16<true>(dr, (uint32_t)(pass * kWave + lane) * 16, w);
        }
        wave_sync();
    };

    const int64_t first = (int64_t)blockIdx.x * kMlpWaves + wave;
    int64_t tile = first;
    fetch(tile);
    flush(-1);
    for (; tile < ntiles; tile += stride) {
        half8_t xc[KC], gc[KC];
#pragma unroll
        for (int s = 0; s < KC; ++s) {
            xc[s] = xn[s];
            gc[s] = gn[s];
        }
        fetch(tile + stride);
        flush(tile != first ? (tile - stride) * 32 : -1);
        __builtin_amdgcn_sched_barrier(0);

        // x and g into the tiles as fetched; back as the lane's own row (chunks hl and 2 + hl: the operands of the
        // per-voxel products) and transposed
        *reinterpret_cast<half8_t*>(xt + foff) = xc[0];
        *reinterpret_cast<half8_t*>(xt + 1024 + foff) = xc[1];
        *reinterpret_cast<half8_t*>(gt + foff) = gc[0];
        *reinterpret_cast<half8_t*>(gt + 1024 + foff) = gc[1];
        wave_sync();
        xc[0] = *reinterpret_cast<const half8_t*>(xt + woff0);
        xc[1] = *reinterpret_cast<const half8_t*>(xt + woff1);
        gc[0] = *reinterpret_cast<const half8_t*>(gt + woff0);
        gc[1] = *reinterpret_cast<const half8_t*>(gt + woff1);
        half8_t xT[2], gT[2];  // lane = channel, registers = voxels 16 hf + 8 hl + 0..7
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            xT[hf] = read_T(xt, hf);
            gT[hf] = read_T(gt, hf);
        }

        float16_t dacc;  // dx^T: D[c][v]
#pragma unroll
        for (int i = 0; i < 16; ++i) dacc[i] = 0.0f;

            // (measurement switch: -DKEROPS_MLP_MH=0 builds the kernel without its arithmetic, i.e. the time of its
            // memory traffic alone: 0.56 ms at (1,32,350,350,128) against 0.61 ms with the arithmetic; two more tiles
            // in flight per wavefront change neither, half as many wavefronts per compute unit bring the traffic
            // alone to 0.52 ms and the whole kernel to 0.69 ms)
#ifndef KEROPS_MLP_MH
#define KEROPS_MLP_MH MH
#endif
#pragma unroll
        for (int mh = 0; mh < KEROPS_MLP_MH; ++mh) {
            float16_t up, dn;
#pragma unroll
            for (int i = 0; i < 16; ++i) up[i] = dn[i] = 0.0f;
#pragma unroll
            for (int s = 0; s < KC; ++s) {
                up = __builtin_amdgcn_mfma_f32_32x32x16_f16(f1[(mh * KC + s) * 64], xc[s], up, 0, 0, 0);
                dn = __builtin_amdgcn_mfma_f32_32x32x16_f16(f2[(mh * KC + s) * 64], gc[s], dn, 0, 0, 0);
            }
            // up[i], dn[i]: hidden channel 32 mh + 8 (i/4) + 4 hl + i%4 of voxel il
            half8_t hv[2], lv[2];
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                const half4_t b4 = *reinterpret_cast<const half4_t*>(bsh + 32 * mh + 8 * gq + 4 * hl);
#pragma unroll
                for (int jp = 0; jp < 2; ++jp) {
                    const int i = 4 * gq + 2 * jp, e = 4 * (gq % 2) + 2 * jp;
                    half2_t hid, lg;
                    hid_lg_pair(up[i], up[i + 1], dn[i], dn[i + 1], half2_t{b4[2 * jp], b4[2 * jp + 1]}, hid, lg);
                    hv[gq / 2][e] = hid[0];
                    hv[gq / 2][e + 1] = hid[1];
                    lv[gq / 2][e] = lg[0];
                    lv[gq / 2][e + 1] = lg[1];
                }
            }
            // rows past V hold x = g = 0: hid = relu(bias) there meets g = 0 in dWdown, lg = 0 everywhere else
            dacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f3[(2 * mh) * 64], lv[0], dacc, 0, 0, 0);
            dacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f3[(2 * mh + 1) * 64], lv[1], dacc, 0, 0, 0);

            // hid and lg rows of the voxel (positions 8 (2 f + hl) + e) into the tiles, back transposed
            wave_sync();  // (the reads of the previous block are issued)
            *reinterpret_cast<half8_t*>(ht + woff0) = hv[0];
            *reinterpret_cast<half8_t*>(ht + woff1) = hv[1];
            *reinterpret_cast<half8_t*>(lt + woff0) = lv[0];
            *reinterpret_cast<half8_t*>(lt + woff1) = lv[1];
            wave_sync();
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const half8_t hT = read_T(ht, hf), lT = read_T(lt, hf);  // lane = hidden position il
                wdn[mh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hT, gT[hf], wdn[mh], 0, 0, 0);
                wup[mh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xT[hf], lT, wup[mh], 0, 0, 0);
                bacc[mh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, lT, bacc[mh], 0, 0, 0);
            }
        }

        // ---- dx: row il of the wavefront's tile, 8 bytes (channels 8 gq + 4 hl + 0..3) at a time; the two halves
        // of a chunk are swapped in every second group of eight rows so that the 16 lanes of a write phase hit 16
        // different pairs of the 32 write banks ----
#pragma unroll
        for (int gq = 0; gq < C / 8; ++gq) {
            half4_t o;
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) o[jj] = (half_t)dacc[4 * gq + jj];
            *reinterpret_cast<half4_t*>(dt + il * 64 + ((gq ^ wsw) * 16) + ((hl ^ ((il >> 3) & 1)) * 8)) = o;
        }
        wave_sync();
    }
    if (first < ntiles) flush((tile - stride) * 32);

    // ---- the four wavefronts add their partials in LDS, wavefront 0 first: [dWup C*H][dWdown H*C][dbias H] ----
    float* red = reinterpret_cast<float*>(smem);
    __syncthreads();  // every wavefront is done with the fragments
#pragma unroll 1
    for (int w = 0; w < kMlpWaves; ++w) {
        if (wave == w) {
#pragma unroll
            for (int mh = 0; mh < MH; ++mh) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int ri = 8 * (i / 4) + 4 * hl + i % 4;  // row of the block held in register i
                    {  // dWdown[h = 32 mh + hidden of position ri][c = il]
                        float* p = red + C * H + (32 * mh + tr_hidden(ri)) * C + il;
                        *p = w == 0 ? wdn[mh][i] : *p + wdn[mh][i];
                    }
                    {  // dWup[c = ri][h = 32 mh + hidden of position il]
                        float* p = red + ri * H + 32 * mh + tr_hidden(il);
                        *p = w == 0 ? wup[mh][i] : *p + wup[mh][i];
                    }
                }
                if (lane < 16) {  // rows 0 and 1 of the 16x16 block: hidden positions lane and 16 + lane
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        float* p = red + 2 * C * H + 32 * mh + tr_hidden(16 * r + lane);
                        *p = w == 0 ? bacc[mh][r] : *p + bacc[mh][r];
                    }
                }
            }
        }
        __syncthreads();
    }
    float* out = ws + (int64_t)blockIdx.x * Cfg::RW;
    for (int i = t; i < Cfg::RW; i += kMlpThreads) out[i] = red[i];
}

// sums the rows of the partial buffer in a fixed order (sum_lines in common.hpp) and scatters the three results
// (OutT: fp32, or fp16 = the fp32 results rounded once)
template <class OutT>
__global__ __launch_bounds__(1024) void mlp_reduce_kernel(const float* __restrict__ ws, int nrows, int RW, int n_up,
                                                          int n_down, OutT* __restrict__ d_up,
                                                          OutT* __restrict__ d_down, OutT* __restrict__ d_bias)
{
    __shared__ double part[16][33];
    const double v = sum_lines(ws, nrows, RW, part);
    const int j = blockIdx.x * 32 + threadIdx.x;
    if (threadIdx.x < 32) {
        if (j < n_up) d_up[j] = (OutT)(float)v;
        else if (j < n_up + n_down) d_down[j - n_up] = (OutT)(float)v;
        else d_bias[j - n_up - n_down] = (OutT)(float)v;
    }
}

static void launch_mlp_reduce(const float* ws, int nrows, int RW, int n_up, int n_down, void* d_up, void* d_down,
                              void* d_bias, int dtype, hipStream_t s)
{
    if (dtype == KEROPS_DTYPE_F16)
        hipLaunchKernelGGL(mlp_reduce_kernel<half_t>, dim3(RW / 32), dim3(1024), 0, s, ws, nrows, RW, n_up,
                           n_down, (half_t*)d_up, (half_t*)d_down, (half_t*)d_bias);
    else
        hipLaunchKernelGGL(mlp_reduce_kernel<float>, dim3(RW / 32), dim3(1024), 0, s, ws, nrows, RW, n_up,
                           n_down, (float*)d_up, (float*)d_down, (float*)d_bias);
}

// workgroups and partial rows per workgroup
static int mb_blocks(int64_t V, int C)
{
    if (C <= 32) {  // wavefront-per-tile kernel: as many workgroups per compute unit as its registers allow
        const int64_t ntiles = (V + 31) / 32;
        return (int)std::max<int64_t>(1, std::min<int64_t>((ntiles + kMlpWaves - 1) / kMlpWaves, C == 16 ? 768 : 512));
    }
    return (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div64(V, MbCfg::TILE), 2 * device_geometry().cus));
}

}  // namespace kerops

extern "C" int64_t kerops_lin_brelu_lin_bwd_workspace_bytes(int64_t V, int32_t C)
{
    if (V <= 0) {
        set_error("lin_brelu_lin_bwd: non-positive size");
        return KEROPS_E_BADARG;
    }
    if (!(C == 16 || C == 32 || C == 64)) {
        set_error("lin_brelu_lin_bwd: built for C in {16,32,64} (got %d)", C);
        return KEROPS_E_UNSUPPORTED_C;
    }
    return (int64_t)mb_blocks(V, C) * (4 * C * C + 2 * C) * (int64_t)sizeof(float);
}

extern "C" int kerops_lin_brelu_lin_bwd_f16(const void* x, const void* g, const void* Wup, const void* Wdown,
                                            const void* bias, void* dx, float* dWup, float* dWdown, float* dbias,
                                            void* workspace, int64_t workspace_bytes, int64_t V, int32_t C,
                                            void* stream)
{
    return kerops_lin_brelu_lin_bwd_f16_out(x, g, Wup, Wdown, bias, dx, dWup, dWdown, dbias, KEROPS_DTYPE_F32, workspace,
                                            workspace_bytes, V, C, stream);
}

extern "C" int kerops_lin_brelu_lin_bwd_f16_out(const void* x, const void* g, const void* Wup, const void* Wdown,
                                                const void* bias, void* dx, void* dWup, void* dWdown, void* dbias,
                                                int32_t grad_dtype, void* workspace, int64_t workspace_bytes, int64_t V,
                                                int32_t C, void* stream)
{
    if (!grad_dtype_ok(grad_dtype)) {
        set_error("lin_brelu_lin_bwd: grad_dtype must be KEROPS_DTYPE_F32 or KEROPS_DTYPE_F16");
        return KEROPS_E_BADARG;
    }
    const int64_t need = kerops_lin_brelu_lin_bwd_workspace_bytes(V, C);
    if (need < 0) return (int)need;
    if (!x || !g || !Wup || !Wdown || !bias || !dx || !dWup || !dWdown || !dbias || !aligned16(x) || !aligned16(g) ||
        !aligned16(Wup) || !aligned16(Wdown) || !aligned16(dx)) {
        set_error("lin_brelu_lin_bwd: null or misaligned pointer");
        return KEROPS_E_BADARG;
    }
    if (!workspace || !aligned16(workspace) || workspace_bytes < need) {
        set_error("lin_brelu_lin_bwd: workspace of %lld bytes required, %lld given", (long long)need,
                  (long long)workspace_bytes);
        return KEROPS_E_WORKSPACE;
    }
    const int blocks = mb_blocks(V, C);
    hipStream_t s = (hipStream_t)stream;
    float* ws = (float*)workspace;
#define KEROPS_MT_CASE(CV)                                                                                        \
    if (C == CV) {                                                                                                \
        hipLaunchKernelGGL((lin_brelu_lin_bwd_wave_kernel<CV>), dim3(blocks), dim3(kMlpThreads), 0, s,           \
                           (const half_t*)x, (const half_t*)g, (const half_t*)Wup, (const half_t*)Wdown,         \
                           (const half_t*)bias, (half_t*)dx, ws, V);                                             \
        int rc = check_launch("lin_brelu_lin_bwd");                                                               \
        if (rc != KEROPS_OK) return rc;                                                                           \
        const int RW = MtCfg<CV>::RW;                                                                             \
        launch_mlp_reduce(ws, blocks, RW, 2 * CV * CV, 2 * CV * CV, dWup, dWdown, dbias, grad_dtype, s);          \
        return check_launch("lin_brelu_lin_bwd_reduce");                                                          \
    }
    KEROPS_MT_CASE(16)
#ifdef KEROPS_MLP_BWD32_IDENTITY  // (comparison build: the identity-product transposes at C = 32 as well)
    KEROPS_MT_CASE(32)
#endif
#undef KEROPS_MT_CASE
    if (C == 32) {
        hipLaunchKernelGGL(lin_brelu_lin_bwd_tr_kernel, dim3(blocks), dim3(kMlpThreads), 0, s, (const half_t*)x,
                           (const half_t*)g, (const half_t*)Wup, (const half_t*)Wdown, (const half_t*)bias, (half_t*)dx,
                           ws, V);
        int rc = check_launch("lin_brelu_lin_bwd");
        if (rc != KEROPS_OK) return rc;
        const int RW = MrCfg::RW;
        launch_mlp_reduce(ws, blocks, RW, 2 * 32 * 32, 2 * 32 * 32, dWup, dWdown, dbias, grad_dtype, s);
        return check_launch("lin_brelu_lin_bwd_reduce");
    }
    if (C == 64) {
        hipLaunchKernelGGL(lin_brelu_lin_bwd_kernel, dim3(blocks), dim3(kMlpThreads), 0, s, (const half_t*)x,
                           (const half_t*)g, (const half_t*)Wup, (const half_t*)Wdown, (const half_t*)bias, (half_t*)dx,
                           ws, V);
        int rc = check_launch("lin_brelu_lin_bwd");
        if (rc != KEROPS_OK) return rc;
        const int RW = MbCfg::RW;
        launch_mlp_reduce(ws, blocks, RW, 2 * 64 * 64, 2 * 64 * 64, dWup, dWdown, dbias, grad_dtype, s);
        return check_launch("lin_brelu_lin_bwd_reduce");
    }
    set_error("lin_brelu_lin_bwd: built for C in {16,32,64} (got %d)", C);
    return KEROPS_E_UNSUPPORTED_C;
}
