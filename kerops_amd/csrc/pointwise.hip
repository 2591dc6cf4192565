// Pointwise (1x1x1) channel mixing on the matrix cores (gfx950):
//
//   out[v, co] = fp16( sum_ci act(x[v, ci]) * Wm[ci, co] )  (+ add[v, co] in fp16)
//
// x is [V][CIN] fp16 (the memory of a channels_last_3d activation), Wm is [CIN][COUT] fp16.
// The op moves 2*V*(CIN + COUT) bytes and does only 2*V*CIN*COUT flops: it is HBM-bound, the
// matrix cores are used so that the arithmetic never shows up next to the memory stream.
//
// Each wavefront owns tiles of 32 voxels.  The product is computed transposed,
// out^T[co, v] = Wm^T[co, :] . x^T[:, v], with v_mfma_f32_32x32x16_f16: the A operand is a
// 32-row block of Wm^T (16-byte fragments pre-arranged in LDS, one ds_read_b128 per instruction), the
// B operand is x^T, whose per-lane fragment "8 consecutive k of voxel lane%32" is simply one 16-byte
// chunk of the voxel's channel vector: lane half h = lane/32 takes chunk 2s+h in step s.
// The fp32 result fragment of a lane is 4 consecutive output channels
// of one voxel (x 4 row groups x COUT/32 blocks); it is rounded to fp16, bounced through a
// wavefront-private LDS tile [32][COUT] and written back as 16-byte chunks, coalesced, with
// the optional fp16 residual add and the optional running max|out| fused into that pass.
#include "common.hpp"

namespace kerops {

typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kPwThreads = 256;
constexpr int kPwWaves = kPwThreads / kWave;

template <int CIN, int COUT>
struct PwCfg {
    static constexpr int MT = (COUT + 31) / 32;      // 32-row blocks of output channels
    static constexpr int KS = CIN / 16;              // MFMA steps (k = 16 each) = 16-byte chunks a lane loads per voxel
    static constexpr int TILE_HALVES = 32 * COUT;    // dense rows, swizzled: BounceTile in common.hpp
    static constexpr int OUT_CHUNKS = 32 * COUT / 8; // 16-byte chunks of one output tile
    static_assert(CIN % 16 == 0 && CIN <= 128, "CIN in {16,32,64,128}");
    static_assert(COUT % 16 == 0 && COUT <= 128, "COUT in {16,32,64,128}");
    // Workgroups per compute unit of the persistent loop: as few as keep the memory pipe full, which also have the fewest
    // prologues.  With a residual two, at 16 -> 16, whose tiles have the fewest bytes, three (us with 2 / 3 / 4: 16 -> 16 at
    // 0.9 M voxels 16.3 / 15.7 / 15.8, 32 -> 32 at 0.9 M 29.7 / 31.4 / 31.4 and at 4 M 126 / 136 / 139, 64 -> 32 at 2 M
    // 84.8 / 91.3 / 89.9, 64 -> 128 at 0.9 M 99.0 / 100.2 / 99.3).
    // Large volumes run at the memory's rate whatever the number, and then the order of reads and writes counts: some pairs
    // are the fastest with another number, or where a wavefront waits for its stores before it goes on (`drain`), reading and
    // writing in turns as with a condition around every store.  us with the choice above / this one:
    //   16 -> 16 at 16 M 261 / 250, 30 M 505 / 480; 16 -> 32 at 30 M 938 / 900; 16 -> 64 at 8 M 409 / 407, 16 M 883 / 843;
    //   32 -> 64 at 8 M 472 / 467, 16 M 924 / 916; 32 -> 16 at 2 M 44.2 / 43.1, 16 M 365 / 349; 64 -> 32 with the batch-norm map at
    //   4 M 173 / 172, 16 M 741 / 726; 64 -> 64 at 4 M 261 / 257, 8 M 543 / 523; 128 -> 16 at 2 M 123 / 122, 8 M 491 / 487;
    //   128 -> 32 at 2 M 136 / 134, 8 M 573 / 563
    struct Large {
        int64_t from;  // voxels
        int per_cu;
        bool drain;
    };
    static constexpr int64_t kVoxels = 1000;
    static constexpr Large large()
    {
        if (CIN == 16 && COUT == 16) return {6000 * kVoxels, 2, false};
        if (CIN == 16 && COUT == 32) return {12000 * kVoxels, 3, true};
        if (CIN == 16 && COUT == 64) return {3000 * kVoxels, 3, false};
        if (CIN == 32 && COUT == 64) return {6000 * kVoxels, 3, false};
        if (CIN == 32 && COUT == 16) return {700 * kVoxels, 3, true};
        if (CIN == 64 && COUT == 32) return {3000 * kVoxels, 2, true};
        if (CIN == 64 && COUT == 64) return {3000 * kVoxels, 3, false};
        if (CIN == 128 && COUT == 16) return {1500 * kVoxels, 2, true};
        if (CIN == 128 && COUT == 32) return {700 * kVoxels, 3, false};
        return {INT64_MAX, 0, false};
    }
    static bool drains(int64_t V, bool add) { return add && large().drain && V >= large().from; }
    // Without a residual a tile has half the bytes: four, where their LDS fits (64 -> 128, 0.1 M voxels 16.1 with four,
    // 13.2 with the three that fit, 4 M 284 and 285; 128 -> 128 24.3 with four, 18.6 with the two that fit, 4 M 387 and 391).
    static constexpr int LDS_BYTES = kPwWaves * TILE_HALVES * 2 + MT * KS * 64 * 16 + 2 * CIN * 4 + 64;
    static constexpr int FITS = 160 * 1024 / LDS_BYTES;
    static int64_t workgroups(int64_t V, bool add)
    {
        const int per_cu = !add ? (FITS < 4 ? FITS : 4) : V >= large().from ? large().per_cu : CIN + COUT == 32 ? 3 : 2;
        return std::max<int64_t>(1, std::min<int64_t>(ceil_div64(V, 32 * kPwWaves), (int64_t)per_cu * device_geometry().cus));
    }
};

// AFFINE: x is first mapped to fp16(max(fma(x, scale[c], shift[c]), 0)), the arithmetic of the batch-norm + ReLU
// stream op, so that op and the product run as one pass and its result never reaches memory.
template <int CIN, int COUT, bool RELU_IN, bool HAS_ADD, bool ABSMAX, bool AFFINE = false>
__global__ __launch_bounds__(kPwThreads) void pointwise_kernel(const half_t* __restrict__ x,
                                                               const half_t* __restrict__ Wm,
                                                               const half_t* __restrict__ add,
                                                               half_t* __restrict__ out, float* __restrict__ amax_ws,
                                                               int64_t V, const float* __restrict__ scale,
                                                               const float* __restrict__ shift, int drain)
{
    using Cfg = PwCfg<CIN, COUT>;
    constexpr int MT = Cfg::MT, KS = Cfg::KS;
    using Tile = BounceTile<COUT>;
    __shared__ __attribute__((aligned(16))) half_t tile[kPwWaves][Cfg::TILE_HALVES];
    __shared__ __attribute__((aligned(16))) half_t wfrag[MT * KS * 64 * 8];
    __shared__ float red[kPwWaves];
    __shared__ __attribute__((aligned(16))) float aff[AFFINE ? 2 * CIN : 4];  // [scale | shift]

    const int t = threadIdx.x, lane = t % kWave, wave = __builtin_amdgcn_readfirstlane(t / kWave);
    const int vl = lane % 32, hl = lane / 32;
    const half8_t z8 = {0, 0, 0, 0, 0, 0, 0, 0};

    // The rows of Wm, 16 bytes at a time and all at once; they go to LDS behind the first tile's loads: one trip to memory
    // for both (two-byte loads ahead of everything else: 32 -> 32 at 50000 voxels with residual 5.1 us, now 4.0; 64 -> 128
    // 11.5, 8.2; 128 -> 128 15.8, 12.4).
    constexpr int NWC = CIN * COUT / 8, NLW = (NWC + kPwThreads - 1) / kPwThreads;
    const plane_rsrc_t wr = plane_rsrc(Wm, CIN * COUT * 2);
    half8_t wpre[NLW];
#pragma unroll
    for (int i = 0; i < NLW; ++i) wpre[i] = plane_load16<false>(wr, (uint32_t)(t + i * kPwThreads) * 16);

    float amax = 0.0f;
    const int64_t ntiles = (V + 31) / 32;
    const int64_t tiles_per_round = (int64_t)gridDim.x * kPwWaves;
    const int64_t nrounds = (ntiles + tiles_per_round - 1) / tiles_per_round;
    unsigned char* my = reinterpret_cast<unsigned char*>(tile[wave]);

    // The tile's part of a tensor with `row` bytes per voxel: nothing stands behind a condition and the compiler's waits are
    // exact, a tile's x fragments are waited for with the stores of the one before in flight.
    auto tile_rsrc = [&](const half_t* p, int64_t tidx, int row) { return rows_rsrc(p, tidx * 32, 32, V, row); };
    // B fragments of a tile: this lane's voxel, chunks 2q+hl
    half8_t xb[KS], xn[KS];
    auto load_x = [&](int64_t tidx, half8_t(&xb)[KS]) {
        const plane_rsrc_t r = tile_rsrc(x, tidx, 2 * CIN);
        // a load instruction touches 32 bytes of every voxel row: rows of 128 bytes and more need the cache to hold the
        // line until the row's other loads arrive, so only narrow rows stream
#pragma unroll
        for (int q = 0; q < KS; ++q) xb[q] = plane_load16<(CIN <= 32)>(r, (uint32_t)(vl * 2 * CIN + 16 * (2 * q + hl)));
    };
    // residual chunks of a tile, in the order in which the results leave the LDS tile
    constexpr int NC = Cfg::OUT_CHUNKS / kWave;
    half8_t ab[HAS_ADD ? NC : 1];
    // Without a residual the loads of the next tile are issued before this tile's arithmetic and stores.  With one they
    // are issued as soon as this tile has used its registers: the x fragments behind the matrix instructions, a residual
    // chunk behind the store of its sum.  Both streams of a tile are then in flight while the previous one is stored.
    // (Loading a residual chunk where it is added costs one memory latency per chunk: 64 -> 128 channels with residual
    // at 0.88 M voxels 130 us, now 103, i.e. 4.4 and 5.5 TB/s; 128 -> 128 at 0.26 M 54 and 39 us.)
    const int64_t first = (int64_t)blockIdx.x * kPwWaves + wave;
    load_x(first, xb);
    // (with the loads and stores in the order of the loop, stores of nothing, so that the waits are the same on both ways
    // into it)
    {
        const plane_rsrc_t ar = tile_rsrc(add, first, 2 * COUT);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            plane_store16<true>(plane_rsrc(out, 0u), 0u, z8);
            if constexpr (HAS_ADD) ab[k] = plane_load16<true>(ar, (uint32_t)(k * kWave + lane) * 16);
        }
    }
    // A fragments: wfrag[((mt*KS + s)*64 + l)*8 + j] = Wm[16 s + 8 (l/32) + j][32 mt + l%32]; 16 output channels fill half
    // a block, the other half is zero
#pragma unroll
    for (int i = 0; i < NLW; ++i) {
        const int c = t + i * kPwThreads, ci = c * 8 / COUT, co = c * 8 % COUT;
        if (c < NWC) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                wfrag[((co / 32 * KS + ci / 16) * 64 + ci % 16 / 8 * 32 + co % 32 + j) * 8 + ci % 8] = wpre[i][j];
        }
    }
    if constexpr (COUT == 16) {
        for (int i = t; i < KS * 32; i += kPwThreads)
            *reinterpret_cast<half8_t*>(wfrag + ((i / 32 * 64 + i % 32 / 16 * 32 + 16 + i % 16) * 8)) = z8;
    }
    if constexpr (AFFINE) {
        for (int i = t; i < CIN; i += kPwThreads) {
            aff[i] = scale[i];
            aff[CIN + i] = shift[i];
        }
    }
    __syncthreads();
    const half8_t* wa = reinterpret_cast<const half8_t*>(wfrag) + lane;
    for (int64_t r = 0; r < nrounds; ++r) {
        const int64_t tidx = (r * gridDim.x + blockIdx.x) * kPwWaves + wave;
        const int64_t v0 = tidx * 32;
        if (HAS_ADD && drain) wait_all_accesses();  // (uniform)
        if constexpr (!HAS_ADD) load_x(tidx + tiles_per_round, xn);
        {
            if constexpr (AFFINE) {
#pragma unroll
                for (int q = 0; q < KS; ++q) {
                    const int c0 = 8 * (2 * q + hl);  // the chunk's first channel: two addresses per wavefront
                    const float4_t s0 = *reinterpret_cast<const float4_t*>(aff + c0);
                    const float4_t s1 = *reinterpret_cast<const float4_t*>(aff + c0 + 4);
                    const float4_t b0 = *reinterpret_cast<const float4_t*>(aff + CIN + c0);
                    const float4_t b1 = *reinterpret_cast<const float4_t*>(aff + CIN + c0 + 4);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        xb[q][j] = (half_t)fmaxf(__builtin_fmaf((float)xb[q][j], s0[j], b0[j]), 0.0f);
                        xb[q][4 + j] = (half_t)fmaxf(__builtin_fmaf((float)xb[q][4 + j], s1[j], b1[j]), 0.0f);
                    }
                }
            }
            if (RELU_IN) {
#pragma unroll
                for (int q = 0; q < KS; ++q) xb[q] = __builtin_elementwise_max(xb[q], z8);  // packed maximum
            }
            float16_t acc[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[mt][i] = 0.0f;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wa[(mt * KS + s) * 64], xb[s], acc[mt], 0, 0, 0);
            }
            // acc[mt][i]: output channel 32*mt + 8*(i/4) + 4*hl + i%4 of voxel vl
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    const int co = 32 * mt + 8 * gq + 4 * hl;
                    if (co < COUT) {
                        half4_t o;
#pragma unroll
                        for (int j = 0; j < 4; ++j) o[j] = (half_t)acc[mt][4 * gq + j];
                        *reinterpret_cast<half4_t*>(my + Tile::piece(vl, 4 * mt + gq, hl)) = o;
                    }
                }
        }
        if constexpr (HAS_ADD) load_x(tidx + tiles_per_round, xb);
        // the tile is private to the wavefront and its LDS operations complete in issue order: no workgroup
        // barrier, the wavefronts of a workgroup run independently
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const plane_rsrc_t outr = tile_rsrc(out, tidx, 2 * COUT), addr = tile_rsrc(add, tidx + tiles_per_round, 2 * COUT);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const int c = k * kWave + lane;
            const int row = c / (COUT / 8), cc = c % (COUT / 8);
            half8_t o = Tile::read(my, row, cc);
            if constexpr (HAS_ADD) {
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = (half_t)((float)o[j] + (float)ab[k][j]);  // fp16 add, RNE
            }
            if (ABSMAX) {
                const bool inside = v0 + row < V;
#pragma unroll
                for (int j = 0; j < 8; ++j) amax = fmaxf(amax, inside ? fabsf((float)o[j]) : 0.0f);
            }
            plane_store16<true>(outr, (uint32_t)c * 16, o);
            if constexpr (HAS_ADD) ab[k] = plane_load16<true>(addr, (uint32_t)c * 16);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if constexpr (!HAS_ADD) {
#pragma unroll
            for (int q = 0; q < KS; ++q) xb[q] = xn[q];
        }
    }
    if (ABSMAX) {
        amax = wave_max(amax);
        if (lane == 0) red[wave] = amax;
        __syncthreads();
        if (t == 0) {
            float m = red[0];
#pragma unroll
            for (int wv = 1; wv < kPwWaves; ++wv) m = fmaxf(m, red[wv]);
            amax_ws[blockIdx.x] = m;
        }
    }
}

__global__ __launch_bounds__(256) void pw_absmax_final_kernel(const float* __restrict__ ws, int n,
                                                              float* __restrict__ out)
{
    __shared__ float red[4];
    float m = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) m = fmaxf(m, ws[i]);
    m = wave_max(m);
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) out[0] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

int pointwise_blocks(int64_t V)
{
    const int64_t ntiles = (V + 31) / 32;
    int64_t b = (ntiles + kPwWaves - 1) / kPwWaves;
    if (b > 1024) b = 1024;  // 4 workgroups of 4 wavefronts per CU, each looping over tiles
    return (int)std::max<int64_t>(b, 1);
}

template <int CIN, int COUT>
static int launch_pw(const half_t* x, const half_t* Wm, const half_t* add, half_t* out, float* amax_ws, int64_t V,
                     bool relu_in, bool absmax, hipStream_t s, const float* scale, const float* shift)
{
    if (absmax && (add || scale)) {  // no instantiation keeps the running max next to a residual or the affine map
        set_error("pointwise: the running max is built without residual add and without the affine map");
        return KEROPS_E_BADARG;
    }
    const int blocks = absmax ? pointwise_blocks(V) : (int)PwCfg<CIN, COUT>::workgroups(V, add != nullptr);
    const int drain = PwCfg<CIN, COUT>::drains(V, add != nullptr);
    if (scale) {  // the affine map ends in a ReLU of its own
        if (add) {
            hipLaunchKernelGGL((pointwise_kernel<CIN, COUT, false, true, false, true>), dim3(blocks), dim3(kPwThreads), 0,
                               s, x, Wm, add, out, amax_ws, V, scale, shift, drain);
        } else {
            hipLaunchKernelGGL((pointwise_kernel<CIN, COUT, false, false, false, true>), dim3(blocks), dim3(kPwThreads),
                               0, s, x, Wm, add, out, amax_ws, V, scale, shift, drain);
        }
        return check_launch("bnrelu_pointwise");
    }
#define KEROPS_PW_GO(R, A, M)                                                                                    \
    hipLaunchKernelGGL((pointwise_kernel<CIN, COUT, R, A, M>), dim3(blocks), dim3(kPwThreads), 0, s, x, Wm, add, \
                       out, amax_ws, V, nullptr, nullptr, drain)
    if (absmax) {
        if (relu_in) KEROPS_PW_GO(true, false, true);
        else KEROPS_PW_GO(false, false, true);
    } else if (add) {
        if (relu_in) KEROPS_PW_GO(true, true, false);
        else KEROPS_PW_GO(false, true, false);
    } else {
        if (relu_in) KEROPS_PW_GO(true, false, false);
        else KEROPS_PW_GO(false, false, false);
    }
#undef KEROPS_PW_GO
    return check_launch("pointwise");
}

int pointwise_dispatch(const half_t* x, const half_t* Wm, const half_t* add, half_t* out, float* amax_ws, int64_t V,
                       int Cin, int Cout, bool relu_in, bool absmax, hipStream_t s, const float* scale, const float* shift)
{
#define KEROPS_PW_CASE(CI, CO)      \
    if (Cin == CI && Cout == CO)    \
        return launch_pw<CI, CO>(x, Wm, add, out, amax_ws, V, relu_in, absmax, s, scale, shift);
    KEROPS_PW_CASE(16, 16)
    KEROPS_PW_CASE(16, 32)
    KEROPS_PW_CASE(32, 16)
    KEROPS_PW_CASE(32, 32)
    KEROPS_PW_CASE(64, 16)
    KEROPS_PW_CASE(64, 32)
    KEROPS_PW_CASE(64, 64)
    KEROPS_PW_CASE(64, 128)
    KEROPS_PW_CASE(128, 16)
    KEROPS_PW_CASE(128, 32)
    KEROPS_PW_CASE(128, 64)
    KEROPS_PW_CASE(128, 128)
    KEROPS_PW_CASE(16, 64)
    KEROPS_PW_CASE(32, 64)
    KEROPS_PW_CASE(16, 128)
    KEROPS_PW_CASE(32, 128)
#undef KEROPS_PW_CASE
    set_error("pointwise: no kernel built for Cin=%d Cout=%d (both in {16,32,64,128})", Cin, Cout);
    return KEROPS_E_UNSUPPORTED_C;
}

void launch_pw_absmax_final(const float* ws, int n, float* out, hipStream_t s)
{
    hipLaunchKernelGGL(pw_absmax_final_kernel, dim3(1), dim3(256), 0, s, ws, n, out);
}

}  // namespace kerops

using namespace kerops;

extern "C" int kerops_pointwise_f16(const void* x, const void* Wm, const void* add, void* out, int64_t V, int32_t Cin,
                                    int32_t Cout, int32_t relu_in, void* stream)
{
    if (!x || !Wm || !out || !aligned16(x) || !aligned16(Wm) || !aligned16(out) || (add && !aligned16(add))) {
        set_error("pointwise: null or misaligned pointer");
        return KEROPS_E_BADARG;
    }
    if (V <= 0) {
        set_error("pointwise: V must be positive");
        return KEROPS_E_BADARG;
    }
    return pointwise_dispatch((const half_t*)x, (const half_t*)Wm, (const half_t*)add, (half_t*)out, nullptr, V, Cin,
                              Cout, relu_in != 0, false, (hipStream_t)stream);
}

extern "C" int kerops_bnrelu_pointwise_f16(const void* x, const float* scale, const float* shift, const void* Wm,
                                           const void* add, void* out, int64_t V, int32_t Cin, int32_t Cout,
                                           void* stream)
{
    if (!x || !scale || !shift || !Wm || !out || !aligned16(x) || !aligned16(Wm) || !aligned16(out) ||
        (add && !aligned16(add))) {
        set_error("bnrelu_pointwise: null or misaligned pointer");
        return KEROPS_E_BADARG;
    }
    if (V <= 0) {
        set_error("bnrelu_pointwise: V must be positive");
        return KEROPS_E_BADARG;
    }
    return pointwise_dispatch((const half_t*)x, (const half_t*)Wm, (const half_t*)add, (half_t*)out, nullptr, V, Cin,
                              Cout, false, false, (hipStream_t)stream, scale, shift);
}
