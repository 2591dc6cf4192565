// Shared device/host helpers for the gfx950 kernels of kerops_amd.
//
// Data layout everywhere: a torch (N, C, H, W, D) channels_last_3d tensor is the
// dense array [N][H][W][D][C] of fp16; D is the innermost spatial axis and the
// C channels of one voxel are contiguous (2*C bytes).  All kernels move data as
// 16-byte chunks of 8 consecutive channels ("c8 chunks"): consecutive lanes of a
// 64-wide wavefront take consecutive chunks, so every global access of a
// wavefront is one contiguous 1 KiB run.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <type_traits>

#include "../../include/kerops_hip.h"

namespace kerops {

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

// An fp32 result that is about to be rounded to fp16, made opaque to the compiler.  Where results are specified as
// fp16(fp32 value) (two roundings, what the reference's kernels and the oracle compute), the product or fused
// multiply-add must exist as an fp32 value first: left alone, the compiler may merge it with the conversion into
// v_fma_mixlo_f16 / v_fma_mixhi_f16, which round the exact result once and differ in the last bit in rare cases.
__device__ __forceinline__ float as_fp32_value(float f)
{
    asm("" : "+v"(f));
    return f;
}
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// ---- shared by the matrix-core depthwise kernels (v_mfma_f32_4x4x4_16B_f16, one block per channel) ----
// LDS patches keep one position in PB = 2*channels bytes; inside a position the channel offset is
// rotated by 32 bytes per position so that the three or four distinct positions read by half a
// wavefront (8 channel pairs each) fall into disjoint banks.  p may be taken relative to any multiple of 4.
template <int PB>
__device__ constexpr int lds_swizzle(int p, int cb)
{
    return p * PB + ((cb + (PB >= 64 ? 32 * (p / (128 / PB)) : 0)) & (PB - 1));
}
// dwords holding two channels at consecutive positions -> the even and the odd channel's fp16x4 operand
__device__ __forceinline__ void split_operands(const uint32_t (&r)[4], half4_t& even, half4_t& odd)
{
    const u32x2_t e = {__builtin_amdgcn_perm(r[1], r[0], 0x05040100u), __builtin_amdgcn_perm(r[3], r[2], 0x05040100u)};
    const u32x2_t o = {__builtin_amdgcn_perm(r[1], r[0], 0x07060302u), __builtin_amdgcn_perm(r[3], r[2], 0x07060302u)};
    even = __builtin_bit_cast(half4_t, e);
    odd = __builtin_bit_cast(half4_t, o);
}
// the same with per-lane byte selectors (0x05040100 / 0x07060302 for live lanes): a lane whose results are never
// used passes 0x0c0c0c0c twice and gets all-zero operands, so that its share of the multipliers does not toggle
__device__ __forceinline__ void split_operands_sel(const uint32_t (&r)[4], uint32_t sel_even, uint32_t sel_odd,
                                                   half4_t& even, half4_t& odd)
{
    const u32x2_t e = {__builtin_amdgcn_perm(r[1], r[0], sel_even), __builtin_amdgcn_perm(r[3], r[2], sel_even)};
    const u32x2_t o = {__builtin_amdgcn_perm(r[1], r[0], sel_odd), __builtin_amdgcn_perm(r[3], r[2], sel_odd)};
    even = __builtin_bit_cast(half4_t, e);
    odd = __builtin_bit_cast(half4_t, o);
}
// same with three positions; the fourth operand element is zero (selector byte 0x0c yields 0x00)
__device__ __forceinline__ void split_operands3(const uint32_t (&r)[3], half4_t& even, half4_t& odd)
{
    const u32x2_t e = {__builtin_amdgcn_perm(r[1], r[0], 0x05040100u), __builtin_amdgcn_perm(0u, r[2], 0x0c0c0100u)};
    const u32x2_t o = {__builtin_amdgcn_perm(r[1], r[0], 0x07060302u), __builtin_amdgcn_perm(0u, r[2], 0x0c0c0302u)};
    even = __builtin_bit_cast(half4_t, e);
    odd = __builtin_bit_cast(half4_t, o);
}

// every lane takes the value of the previous lane of its quad (lane 0 that of lane 3): one DPP move per dword
__device__ __forceinline__ half4_t quad_rotate_up(half4_t v)
{
    u32x2_t w = __builtin_bit_cast(u32x2_t, v);
    // (every lane has a source, so the "old" operand is never kept: passing the source itself lets the move run in place)
    w[0] = (uint32_t)__builtin_amdgcn_update_dpp((int)w[0], (int)w[0], 0x93, 0xf, 0xf, false);  // quad_perm:[3,0,1,2]
    w[1] = (uint32_t)__builtin_amdgcn_update_dpp((int)w[1], (int)w[1], 0x93, 0xf, 0xf, false);
    return __builtin_bit_cast(half4_t, w);
}

constexpr int kWave = 64;

// ---- LDS-direct loads (global_load_lds_dwordx4) with hand-placed waits ------------------------------------
// The compiler neither sees these memory instructions nor counts them: a kernel that uses them issues the same
// number of them in every wavefront and step (an instruction whose mask is empty still counts) and waits with
// wait_loads_in_flight<n>, which returns when all but the newest n vector memory instructions of the wavefront
// have completed (loads and stores retire in issue order).  M0 is used by nothing else in these kernels.
// one LDS-direct load of a wavefront: lane l brings the 16 bytes at sbase + voff to LDS address lds_addr + 16*l;
// lanes outside `mask` do nothing.  sbase, lds_addr and mask are wavefront-uniform (scalar registers).
template <bool STREAM>
__device__ __forceinline__ void lds_direct_load16(const void* sbase, uint32_t voff, uint32_t lds_addr, uint64_t mask)
{
    uint64_t saved;
    if (STREAM)
        asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, %4\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %2, %1 nt\n\ts_mov_b64 exec, %0"
                     : "=&s"(saved)
                     : "s"(sbase), "v"(voff), "s"(lds_addr), "s"(mask)
                     : "memory");
    else
        asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, %4\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %2, %1\n\ts_mov_b64 exec, %0"
                     : "=&s"(saved)
                     : "s"(sbase), "v"(voff), "s"(lds_addr), "s"(mask)
                     : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads_in_flight()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// until every vector memory access of the wavefront has completed (the compiler's own accesses; it sees this wait)
__device__ __forceinline__ void wait_all_accesses() { __builtin_amdgcn_s_waitcnt(0x0f70); }
__device__ __forceinline__ const char* uniform_ptr(const char* p)
{
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const char*>(((uint64_t)hi << 32) | lo);
}

// 16-byte streaming store of the lanes in `mask` to sbase + voff, counted like the loads above
__device__ __forceinline__ void masked_store16_stream(void* sbase, uint32_t voff, u32x4_t data, uint64_t mask)
{
    uint64_t saved;
    asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, %4\n\tglobal_store_dwordx4 %2, %3, %1 nt\n\ts_mov_b64 exec, %0"
                 : "=&s"(saved)
                 : "s"(sbase), "v"(voff), "v"(data), "s"(mask)
                 : "memory");
}

// ---- plane access with the hardware's bounds check ---------------------------------------------------------
// A buffer access whose byte offset is not below the resource's size does nothing: a load returns zeros, a store is
// dropped, no memory is touched.  So a plane that does not exist has size 0 and a lane without a voxel an offset past
// every plane, and no condition stands around the instruction: the compiler's wait-count bookkeeping is exact only on
// branch-free paths (behind a conditional store it waits for every access in flight).
typedef __amdgpu_buffer_rsrc_t plane_rsrc_t;
constexpr uint32_t kNoVoxel = 0xfffffff0u;  // no offset below the bytes of a plane of at most 2^31 - 8 fp16 elements
__device__ __forceinline__ plane_rsrc_t plane_rsrc(const void* plane, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(plane), 0, (int)bytes, 0x27000);
}
template <bool STREAM>
__device__ __forceinline__ half8_t plane_load16(plane_rsrc_t r, uint32_t voff)
{
    return __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, 0, STREAM ? 2 : 0));
}
template <bool STREAM>
__device__ __forceinline__ void plane_store16(plane_rsrc_t r, uint32_t voff, half8_t v)
{
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), r, (int)voff, 0, STREAM ? 2 : 0);
}

// The rows [v0, v0 + rows) of a [V][row_bytes / 2] tensor; rows that do not exist (past V, or v0 < 0) have no bytes, so a
// tile's accesses stand behind no condition.  (v0 wavefront-uniform, rows * row_bytes < 2^31)
__device__ __forceinline__ plane_rsrc_t rows_rsrc(const half_t* p, int64_t v0, int rows, int64_t V, int row_bytes)
{
    const bool some = v0 >= 0 && v0 < V;
    const int n = some ? (int)std::min<int64_t>(V - v0, rows) : 0;
    return plane_rsrc(uniform_ptr(reinterpret_cast<const char*>(p) + (some ? v0 : 0) * row_bytes), (uint32_t)(n * row_bytes));
}

constexpr int64_t kStreamInteriorMinBytes = 384ll << 20;

// Order in which the 16-byte chunks of a staged plane (a TW x TD patch with its one-voxel halo, CG chunks per
// position) are shared out to the threads: first the chunks that a neighbouring patch reads as well (the halo
// ring around the patch and the patch's own border ring), then the interior, which only this workgroup reads.
// A load instruction whose chunks are all interior carries the streaming hint, so these lines do not push the
// shared ones out of the L2 before the neighbour has read them (forward kernel at 64 channels: x fetched from
// memory 1.148 -> 1.108 times, 2.5 % less time; 3 % at 16 channels).  Streaming loads do not use the 256 MB
// memory-side cache either, so the hint is for tensors that cannot stay there anyway: the launchers switch it on
// above kStreamInteriorMinBytes (with the whole 251 MB (1,8,350,350,128) tensor cached between calls the hint cost
// 34 %, with the 268 MB input of the fused block 7 %).  Runs stay whole lines: full rows of TD + 2 positions, pairs
// of positions at the sides, TD - 2 positions inside.
template <int TW, int TD, int CG>
struct HaloOrder {
    static constexpr int ROWCH = (TD + 2) * CG;                  // chunks of one staged row
    static constexpr int NSH_ROWS = 4 * ROWCH;                   // the two rows above and the two below
    static constexpr int NSH = NSH_ROWS + 4 * (TW - 2) * CG;     // ... and two positions at either side
    static constexpr int N = (TW + 2) * ROWCH;
    // chunk index -> staged row wq in [0, TW + 2), position dq in [0, TD + 2), channel chunk cq
    __device__ static __forceinline__ void decode(int ch, int& wq, int& dq, int& cq)
    {
        if (ch < NSH_ROWS) {
            const int r4 = ch / ROWCH, rem = ch - r4 * ROWCH;
            wq = r4 < 2 ? r4 : TW + r4 - 2;
            dq = rem / CG;
            cq = rem - dq * CG;
        } else if (ch < NSH) {
            const int s2 = ch - NSH_ROWS, wr = s2 / (4 * CG), rem = s2 - wr * 4 * CG, dp = rem / CG;
            wq = 2 + wr;
            dq = dp < 2 ? dp : TD + dp - 2;
            cq = rem - dp * CG;
        } else {
            const int pp = ch - NSH, wr = pp / ((TD - 2) * CG), rem = pp - wr * (TD - 2) * CG;
            wq = 2 + wr;
            dq = 2 + rem / CG;
            cq = rem % CG;
        }
    }
    // whether the load that covers the chunks [first, first + count) touches interior chunks only
    static constexpr bool interior_only(int first) { return first >= NSH; }
};

// ---- error reporting (host) -------------------------------------------------
void set_error(const char* fmt, ...);
int check_launch(const char* what);

// ---- device geometry (host) -------------------------------------------------
// Compute units and accelerator dies (XCDs, each with its own L2) of the current device, read once per device
// with hipDeviceGetAttribute (core.hip); without a usable device (a workspace query on a machine without a GPU)
// the MI355X's 256 / 8.  The H-marching kernels size their launch to the workgroups the device holds at once
// and walk every die's share of the tiles contiguously.
struct DeviceGeometry {
    int cus, xcds;
    // workgroups resident at once: 16 wavefronts per compute unit at the register budget of these kernels
    int resident_workgroups(int threads) const { return cus * (threads >= 512 ? 2 : 4); }
};
DeviceGeometry device_geometry();

// ---- cross-file launchers (defined in dwconv_fwd.hip / pointwise.hip) ----------------
int dwconv_fwd_run(const void* x, const void* wt, void* y, const float* scale, const float* shift, int32_t N,
                   int32_t H, int32_t W, int32_t D, int32_t C, int32_t tile_w, int32_t tile_d, int32_t h_chunk,
                   int32_t lane_channels, void* stream);
// fused depthwise -> affine -> ReLU -> pointwise kernel (64 input channels, Cout in {64,128}); workgroup count of
// its grid (= floats of amax_ws it writes)
int dwsep_fused_blocks(int32_t N, int32_t H, int32_t W, int32_t D);
int dwsep_fused_run(const void* x, const void* wt, const float* scale, const float* shift, const void* pw, void* y2,
                    float* amax_ws, int32_t N, int32_t H, int32_t W, int32_t D, int32_t Cout, void* stream);
int pointwise_dispatch(const _Float16* x, const _Float16* Wm, const _Float16* add, _Float16* out, float* amax_ws,
                       int64_t V, int Cin, int Cout, bool relu_in, bool absmax, hipStream_t s,
                       const float* scale = nullptr, const float* shift = nullptr);
int pointwise_blocks(int64_t V);  // workgroups, and maxima in amax_ws, with absmax
void launch_pw_absmax_final(const float* ws, int n, float* out, hipStream_t s);

// ---- small host helpers -----------------------------------------------------
// for a >= 0, b > 0; no intermediate sum, so extents up to the type's maximum are safe
static inline int64_t ceil_div64(int64_t a, int64_t b) { return a / b + (a % b != 0); }
static inline int ceil_div(int a, int b) { return a / b + (a % b != 0); }
static inline bool is_pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }
static inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
// N*H*W*D*C elements (all positive) must be addressable with 64-bit byte offsets; checked before any product
// of extents is formed in 64 bits
static inline bool volume_exceeds_i64(int N, int H, int W, int D, int C)
{
    const __int128 lim = (__int128)1 << 60;
    __int128 v = (__int128)N * H * W;  // < 2^93
    if (v >= lim) return true;
    v *= D;
    if (v >= lim) return true;
    return v * C >= lim;
}
// Rows per workgroup of the H-marching convolution kernels.  All workgroups of a launch do the same work, so
// they run in ceil(workgroups / resident slots) rounds; a workgroup that marches over h rows takes h + 2 plane
// steps (two halo planes) plus a fixed cost of about `setup` plane steps (prologue, pipeline fill, epilogue).
// The split that minimises rounds * (h + 2 + setup) wins; ties go to fewer, longer chunks.  Checked against
// H_chunk sweeps of the forward and weight-gradient kernels at 14 shapes from 96^3 x 16 to 350 x 350 x 128 x 128
// channels: the choice is the sweep's optimum or within 2 % of it (a variant that charges half a round for a
// partial last round instead of a whole one was up to 15 % off).
static inline int pick_h_chunk(int H, int64_t per_plane, int slots, int setup)
{
    int best_h = H;
    double best = 1e300;
    const int max_chunks = H < 64 ? H : 64;
    for (int c = 1; c <= max_chunks; ++c) {
        const int h = ceil_div(H, c);
        const int chunks = ceil_div(H, h);
        if (chunks != c) continue;  // the same split as a smaller c
        const double rounds = std::ceil((double)per_plane * chunks / slots);  // (doubles: no overflow at absurd sizes)
        const double cost = rounds * ((double)h + 2 + setup) * (1.0 + 0.004 * c);
        if (cost < best) {
            best = cost;
            best_h = h;
        }
    }
    return best_h;
}
// Balanced split of the H-marching kernels.  The tiles of the tensor, in their linear order (slab fastest, then
// the tiles along D, along W, the batch), are cut into bundles of `group` neighbours; the launch has `ngroups`
// groups of `group` workgroups, and a group owns a contiguous share of the sequence (bundle, row): its workgroups
// march in step over the tiles of a bundle (they share halo voxels through the L2 of their XCD) and cross into
// the next bundle together.  Every group then carries the same number of plane steps whatever the tile count,
// where uniform chunks leave the last round of workgroups partly filled (2-10 % slower at the shapes measured).
// `row_len` = tiles (times slabs) in one row along D.  The group size is chosen by a cost model fitted to
// sweeps at (1, C, 350, 350, 128), C = 8..128: time ~ plane steps of a group, 10 % / (tile rows in a bundle) for
// the halo rows that neighbouring bundles no longer share in L2, 4 % for a group that does not fit one XCD, a
// fixed cost per workgroup and per crossing.
struct BalancedSplit {
    uint32_t group, ngroups;
    int64_t units;  // bundles * H
};
static inline BalancedSplit make_balanced(int H, int64_t tiles, int slots, int group)
{
    BalancedSplit b;
    b.group = (uint32_t)group;
    const int64_t bundles = tiles / group + (tiles % group != 0);
    // more plane steps than the kernels' 32-bit counters hold: any value >= 2^31 makes the callers fall back
    b.units = bundles > (1LL << 31) / H ? (1LL << 40) : bundles * H;
    // a share of fewer than 2 rows is all halo planes: use fewer groups then
    b.ngroups = (uint32_t)std::min<int64_t>(std::max(1, slots / group), std::max<int64_t>(1, b.units / 2));
    return b;
}
static inline double balanced_cost(const BalancedSplit& b, int H, int row_len, int slots, int setup, int xcds)
{
    const double share = (double)((b.units + b.ngroups - 1) / b.ngroups);
    const double crossings = share / H;  // expected bundle boundaries inside a share
    const double rows = (double)b.group / row_len;
    // a group larger than the workgroups one XCD holds is spread over several L2s (measured: 2-3 % slower)
    const double spread = (int)b.group > slots / xcds ? 1.04 : 1.0;
    return (share + 2 + setup + crossings * 5.0) * (1.0 + 0.1 / rows) * (1.0 + 0.004 * H / share) * spread;
}
// slab_mult: the group size must be a multiple of it (kernels that keep per-slab state across bundles)
template <typename Cost>
static inline BalancedSplit best_balanced(int H, int64_t tiles, int row_len, int slots, int slab_mult, Cost cost,
                                          double* cost_out)
{
    BalancedSplit best = make_balanced(H, tiles, slots, slab_mult);
    double best_cost = 1e300;
    auto consider = [&](int64_t g) {
        if (g < 1 || g > slots || g % slab_mult != 0) return;
        if (g >= tiles + row_len && g > slab_mult) return;  // more than a row of idle members
        const BalancedSplit b = make_balanced(H, tiles, slots, (int)g);
        const double c = cost(b);
        if (c < best_cost) {
            best_cost = c;
            best = b;
        }
    };
    for (int r = 1; r <= 16; ++r) consider((int64_t)r * row_len);             // whole tile rows
    for (int f = 2; f <= 8; f *= 2)                                           // parts of a long row
        if (row_len % f == 0) consider(row_len / f);
    consider(slab_mult);
    *cost_out = best_cost;
    return best;
}
// The split of a launch: the balanced one, or (h_chunk > 0) uniform chunks of h_chunk rows.
// Where a group's share of the balanced split is a whole column of the volume or more, every group crosses into other
// bundles and the cost above decides.  Where it is less, the launch lasts as long as the groups that do cross (two halo
// planes and a pipeline refill), and chunks of equal length without any crossing are often faster although they leave
// workgroup slots empty: the cheaper of the two, with the crossing counted in full, is taken.  Measured over 180
// volumes of 0.26 to 400 M elements, C = 8..128, against the balanced split alone: forward 8.8 % faster on average,
// weight gradient 4.9, fused backward 6.8, between 0.54 and 1.04 of its time ((2,32,96,96,96) forward 55.6 -> 52.7 us,
// (2,128,45,51,37) backward 47.6 -> 43.4, (1,128,34,71,55) forward 24.2 -> 18.5).
struct MarchSplit {
    BalancedSplit b;
    int h_chunk;
};
// What a launch costs beyond its plane steps, per kernel: fitted to every chunk length and a dozen group sizes at 150
// volumes of 0.26 to 240 M elements each.
struct MarchCost {
    int setup;        // plane steps that a workgroup's prologue, pipeline fill and epilogue take
    double crossing;  // plane steps that crossing into another bundle takes
    // A workgroup that has a compute unit of its own steps faster than one of two, so half a round of longer chunks can
    // beat a full round of short ones ((1,64,34,44,29) forward: 408 workgroups of two rows 9.8 us, 216 of four 8.9;
    // fused backward 18.5 and 17.3): the ratio of the two, 1 where it does not pay.
    double alone;
    // Most workgroups that may march over a single row, which reads three planes for one.  Alone on a compute unit such a
    // workgroup is still the faster one ((1,32,33,19,25), 198 of them: forward 6.26 us, 6.60 with two rows each); two of
    // them on a compute unit lose in the forward and weight-gradient kernels ((2,32,32,9,35), 384: forward 8.20 us, 6.81
    // with two rows each, weight gradient 12.2 and 10.9).  The fused backward keeps to single rows wherever they fit, also
    // against the cost below: that was the faster split of its earlier kernel (15.0 and 15.8 us) and is no longer.  Over 36
    // volumes of 257 to 512 such workgroups two rows take 0.90 to 0.95 of its time (the same volume 13.2 and 12.0), over 40
    // of fewer 1.06 to 1.09.  The limit of one workgroup per compute unit would be right here too; it moves together with
    // the test that holds the fused backward's workgroup counts.
    int one_row;
};
static inline MarchSplit pick_split(int H, int64_t tiles, int row_len, int slots, int slab_mult, const DeviceGeometry& geo,
                                    const MarchCost& m)
{
    double cost;
    const BalancedSplit whole = best_balanced(
        H, tiles, row_len, slots, slab_mult,
        [&](const BalancedSplit& b) { return balanced_cost(b, H, row_len, slots, m.setup, geo.xcds); }, &cost);
    if ((whole.units + whole.ngroups - 1) / whole.ngroups >= H) return {whole, 0};
    auto occupancy = [&](int64_t workgroups) { return workgroups <= geo.cus ? m.alone : 1.0; };
    auto part_cost = [&](const BalancedSplit& b) {
        const int64_t share = (b.units + b.ngroups - 1) / b.ngroups;
        const bool aligned = b.units % b.ngroups == 0 && H % share == 0;  // no share crosses
        const double crossing = share < H ? (aligned ? 0.0 : m.crossing) : m.crossing * (double)share / H;
        const double spread = (int)b.group > slots / geo.xcds ? 1.04 : 1.0;
        return ((double)share + 2 + m.setup + crossing) * (1.0 + 0.1 * row_len / (double)b.group) *
               (1.0 + 0.004 * (double)H / (double)share) * spread * occupancy((int64_t)b.group * b.ngroups);
    };
    BalancedSplit part = best_balanced(H, tiles, row_len, slots, slab_mult, part_cost, &cost);
    if (m.alone < 1.0 && geo.cus < slots) {
        double half;
        const BalancedSplit b = best_balanced(H, tiles, row_len, geo.cus, slab_mult, part_cost, &half);
        if (half < cost) {
            cost = half;
            part = b;
        }
    }
    // chunks that run in one round (never more workgroups, and partial sums, than fit the GPU at once)
    int best_h = 0;
    for (int c = 1; c <= 64 && c <= H && tiles * c <= slots; ++c) {
        const int h = ceil_div(H, c);
        if (ceil_div(H, h) != c) continue;  // the same split as a smaller c
        if (h < 2 && c > 1 && tiles * c > m.one_row) break;
        const double uniform = ((double)h + 2 + m.setup) * (1.0 + 0.004 * c) * occupancy(tiles * c);
        if (uniform <= cost || (h == 1 && m.one_row >= slots)) {
            cost = uniform;
            best_h = h;
        }
    }
    return {part, best_h};
}
// offsets inside one (W, D, C) plane are 32-bit in the convolution kernels (W, D, C positive): an element's index is an int,
// its byte offset a uint32_t (doubled as an int it would overflow from 2^30 elements on)
static inline bool plane_exceeds_i32(int W, int D, int C)
{
    const int64_t wd = (int64_t)W * D;  // < 2^62
    return wd >= (1LL << 31) || wd * C >= (1LL << 31);
}

// Device side of the two splits of the H march: the sequence of (tile, rows [hs, he)) segments of one workgroup.
// Tiles are numbered slab fastest, then along D, along W, then the batch.  Uniform chunks (group = 0): one segment,
// workgroup w = (tile inside the sample, chunk, sample).  Balanced split: the workgroup is member w % group of group
// w / group, which owns the units [u, u_end) of the (bundle of `group` tiles, row) sequence; a share that ends inside
// a bundle continues in the next one, and members beyond the last tile of a partly filled bundle skip it.  All
// values are wavefront-uniform and kept in scalar registers.
struct SegmentWalk {
    uint32_t u, u_end, member, group;
    bool first;
};
// shares of q or q + 1 units: the first r groups take the longer ones
__device__ __forceinline__ SegmentWalk segment_walk_begin(uint32_t wg, uint32_t group, uint32_t q, uint32_t r)
{
    SegmentWalk s{0u, 0u, 0u, group, true};
    if (group > 0) {
        const uint32_t g = wg / group;
        s.member = wg - g * group;
        s.u = __builtin_amdgcn_readfirstlane(g * q + min(g, r));
        s.u_end = __builtin_amdgcn_readfirstlane(s.u + q + (g < r ? 1u : 0u));
    }
    return s;
}
__device__ __forceinline__ bool segment_walk_next(SegmentWalk& s, uint32_t wg, int H, uint32_t n_tiles,
                                                  uint32_t tiles_per_sample, int n_hc, int h_chunk, uint32_t& tile,
                                                  int& hs, int& he)
{
    if (s.group > 0) {
        for (;;) {
            if (s.u >= s.u_end) return false;
            const uint32_t bundle = s.u / (uint32_t)H;
            // (the quotient comes out of a vector division: back to scalar registers)
            hs = __builtin_amdgcn_readfirstlane((int)(s.u - bundle * (uint32_t)H));
            he = (int)min((uint32_t)H, hs + (s.u_end - s.u));
            s.u += he - hs;
            tile = __builtin_amdgcn_readfirstlane(bundle * s.group + s.member);
            if (tile < n_tiles) return true;
        }
    }
    if (!s.first) return false;
    s.first = false;
    const uint32_t rest = wg / tiles_per_sample;
    const int hc = (int)(rest % (uint32_t)n_hc);
    tile = __builtin_amdgcn_readfirstlane((rest / (uint32_t)n_hc) * tiles_per_sample + wg % tiles_per_sample);
    hs = __builtin_amdgcn_readfirstlane(hc * h_chunk);
    he = min(hs + h_chunk, H);
    return true;
}

// The XCDs of the chip (8 on MI355X; the launchers pass the device's count) receive workgroups round-robin
// (workgroup b runs on XCD b % n) and each XCD has a private L2.  remap_xcd turns the hardware workgroup
// index into a logical tile index such that each XCD walks one contiguous range of
// logical tiles: neighbouring tiles (which share halo voxels) then meet in the same
// L2 instead of being fetched once per XCD.
__device__ __forceinline__ uint32_t remap_xcd(uint32_t b, uint32_t nblocks, uint32_t n_xcd)
{
    uint32_t per = (nblocks + n_xcd - 1) / n_xcd;  // logical tiles per XCD (last range may be short)
    uint32_t xcd = b % n_xcd;
    uint32_t idx = b / n_xcd;
    // ranges [xcd*per, (xcd+1)*per); the tail ranges can exceed nblocks, so the
    // grid is launched with per*n_xcd workgroups and the caller drops ids >= nblocks.
    return xcd * per + idx;
}
static inline uint32_t xcd_padded_grid(uint32_t nblocks, uint32_t n_xcd) { return ((nblocks + n_xcd - 1) / n_xcd) * n_xcd; }

// ---- 16-byte chunk access ---------------------------------------------------
__device__ __forceinline__ half8_t load_c8(const half_t* p) { return *reinterpret_cast<const half8_t*>(p); }
__device__ __forceinline__ void store_c8(half_t* p, half8_t v) { *reinterpret_cast<half8_t*>(p) = v; }

// Streaming (non-temporal) variants for data that is touched exactly once.
__device__ __forceinline__ half8_t load_c8_nt(const half_t* p)
{
    return __builtin_nontemporal_load(reinterpret_cast<const half8_t*>(p));
}
__device__ __forceinline__ void store_c8_nt(half_t* p, half8_t v)
{
    __builtin_nontemporal_store(v, reinterpret_cast<half8_t*>(p));
}

// ---- LDS tile for results that leave the accumulators in 8-byte pieces and LDS in 16-byte chunks ---------------
// A 32x32x16 accumulator holds, per lane (row = lane % 32, half = lane / 32), groups of four consecutive output
// channels: the 8-byte half `half` of the 16-byte chunk `chunk` of the row.  The rows leave LDS as 16-byte chunks,
// lane c taking chunk c % CPR of row c / CPR, for coalesced stores.  Measured on gfx950, LDS writes see 32 banks of
// 4 bytes (16 lanes of an 8-byte write per clock) and reads 64 (16 lanes of a 16-byte read per clock).  Rows are
// dense (2 * COLS bytes), so the 16 lanes of a read phase take 256 consecutive bytes whatever the order inside a
// row; inside a row the chunk slot and the half are flipped by bits of the row number, chosen so that the 16 rows
// of a write phase (same chunk, same half) fall on 16 different bank pairs.
template <int COLS>
struct BounceTile {
    static constexpr int CPR = COLS / 8, RB = 2 * COLS;     // chunks per row, bytes per row
    static constexpr int RPW = RB >= 128 ? 1 : 128 / RB;    // rows per 128 bytes of write banks
    static constexpr int SW = CPR < 8 ? CPR : 8;            // chunk slots that differ in their write banks
    static constexpr int BYTES = 32 * RB;
    static_assert(COLS == 16 || COLS == 32 || COLS == 64 || COLS == 128, "row widths of the built kernels");
    // byte offset of the 8-byte piece (row, chunk, half)
    __device__ static constexpr int piece(int row, int chunk, int half)
    {
        return row * RB + ((chunk ^ ((row / RPW) % SW)) * 16) + ((half ^ (((row / RPW) / SW) & 1)) * 8);
    }
    // byte offset of the 16-byte chunk (row, chunk); its two halves are swapped where halves_swapped(row)
    __device__ static constexpr int chunk16(int row, int chunk) { return row * RB + ((chunk ^ ((row / RPW) % SW)) * 16); }
    __device__ static constexpr bool halves_swapped(int row) { return (((row / RPW) / SW) & 1) != 0; }
    __device__ static half8_t read(const unsigned char* tile, int row, int chunk)
    {
        const half8_t r = *reinterpret_cast<const half8_t*>(tile + chunk16(row, chunk));
        const bool sw = halves_swapped(row);
        return half8_t{sw ? r[4] : r[0], sw ? r[5] : r[1], sw ? r[6] : r[2], sw ? r[7] : r[3],
                       sw ? r[0] : r[4], sw ? r[1] : r[5], sw ? r[2] : r[6], sw ? r[3] : r[7]};
    }
};

// ---- LDS tile of dense [voxel][channel] fp16 rows that is written as 16-byte chunks, read as 16-byte chunks of
// one voxel (matrix operands with the voxel per lane) and read transposed (operands with the channel per lane) -----
// gfx950 reads LDS transposed: ds_read_b64_tr_b16 takes, in every block of 16 lanes, the 16 x 4 matrix M of 16-bit
// values that the lanes address (lane s supplies the address of four consecutive values M[s][0..3]) and returns to
// lane i the values M[4 j + i/4][i%4], j = 0..3.  With lane s pointing at row s/4, columns 4 (s%4) .. 4 (s%4) + 3
// of a row-major tile, lane i receives column i of four consecutive rows: two such reads make the eight reduction
// values (rows 16 s + 8 (lane/32) + 0..7) of a 32x32x16 operand whose lane index is the column.
// Chunk c of row r sits in chunk slot c ^ slot(r).  slot(r) is chosen so that (measured bank structure: 64 banks
// of 4 bytes for reads, 32 for writes) the 16 rows of a 16-byte read phase that takes the same chunk of each fall
// on different banks, the four rows of a transposing read phase (64 bytes of each) likewise, and writes of whole
// rows are conflict-free by construction.
typedef __attribute__((__vector_size__(4 * sizeof(__fp16)))) __fp16 fp16x4_raw_t;
__device__ __forceinline__ half4_t lds_read_tr16(const unsigned char* p)
{
    const auto q = (__attribute__((address_space(3))) fp16x4_raw_t*)(p);
    return __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4f16(q));
}
template <int COLS>
struct SwizzledRows {
    static constexpr int CPR = COLS / 8, RB = 2 * COLS;
    static_assert(COLS == 16 || COLS == 32 || COLS == 64 || COLS == 128, "row widths of the built kernels");
    __device__ static constexpr int slot(int r)
    {
        return CPR == 2   ? ((r >> 3) & 1)
               : CPR == 4 ? ((r >> 2) & 3)
               : CPR == 8 ? ((((r >> 1) & 1) << 2) | ((r >> 2) & 3))
                          : (((r & 3) << 2) | ((r >> 2) & 3));
    }
    __device__ static constexpr int chunk16(int row, int chunk) { return row * RB + ((chunk ^ slot(row)) * 16); }
    // Per-lane byte offsets of the two transposing reads of reduction step 0 for the 32-column block `blk32`
    // (columns 32 blk32 + lane % 32; a 16-column tile repeats its columns); step s adds s * 16 * RB.
    __device__ static void tr_offsets(int lane, int blk32, int (&off)[2])
    {
        const int s = lane % 16, b16 = COLS >= 32 ? (lane / 16) % 2 : 0, hl = lane / 32;
        const int col = 32 * blk32 + 16 * b16 + 4 * (s % 4);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int row = 8 * hl + 4 * r + s / 4;
            off[r] = chunk16(row, col / 8) + (col % 8) * 2;
        }
    }
    __device__ static half8_t read_tr(const unsigned char* tile, const int (&off)[2], int step)
    {
        const half4_t a = lds_read_tr16(tile + step * 16 * RB + off[0]);
        const half4_t b = lds_read_tr16(tile + step * 16 * RB + off[1]);
        return half8_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    }
};

// ---- wavefront reductions -----------------------------------------------------
// Sum over the lanes of a wavefront whose index differs only in bits >= log2(stride_lo):
// i.e. lanes l and l' are combined when l % stride_lo == l' % stride_lo.
template <int STRIDE_LO>
__device__ __forceinline__ float wave_sum_stride(float v)
{
#pragma unroll
    for (int off = 32; off >= STRIDE_LO; off >>= 1) {
        v += __shfl_xor(v, off, 64);
    }
    return v;
}

__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        v = fmaxf(v, __shfl_xor(v, off, 64));
    }
    return v;
}

}  // namespace kerops

// ---- per-channel streaming helpers (stream_ops.hip, avgpool.hip) --------------
namespace kerops {

// V consecutive fp16 channels moved as one access; V = min(8, C).
template <int V>
struct HVec {
    typedef _Float16 type __attribute__((ext_vector_type(V)));
};
template <>
struct HVec<1> {
    struct type {
        _Float16 s;
        __device__ __forceinline__ _Float16& operator[](int) { return s; }
        __device__ __forceinline__ const _Float16& operator[](int) const { return s; }
    };
};

// Run the statement list with a constexpr `V` = min(8, C) in scope (C a power of two).
#define KEROPS_DISPATCH_V(C, ...)  \
    do {                           \
        if ((C) >= 8) {            \
            constexpr int V = 8;   \
            __VA_ARGS__;           \
        } else if ((C) == 4) {     \
            constexpr int V = 4;   \
            __VA_ARGS__;           \
        } else if ((C) == 2) {     \
            constexpr int V = 2;   \
            __VA_ARGS__;           \
        } else {                   \
            constexpr int V = 1;   \
            __VA_ARGS__;           \
        }                          \
    } while (0)

template <int V>
__device__ __forceinline__ typename HVec<V>::type ld(const _Float16* p, int64_t chunk)
{
    return *reinterpret_cast<const typename HVec<V>::type*>(p + chunk * V);
}
template <int V>
__device__ __forceinline__ void st(_Float16* p, int64_t chunk, const typename HVec<V>::type& v)
{
    *reinterpret_cast<typename HVec<V>::type*>(p + chunk * V) = v;
}
// Streaming variants for data that is touched exactly once by the kernel: the non-temporal hint
// keeps one-pass streams from displacing each other in L2 (measured on MI355X: a pure read
// stream reaches ~6.5 TB/s with the hint against ~5.9 TB/s without).
template <int V>
__device__ __forceinline__ typename HVec<V>::type ld_stream(const _Float16* p, int64_t chunk)
{
    if constexpr (V == 1) {
        return *reinterpret_cast<const typename HVec<V>::type*>(p + chunk * V);
    } else {
        return __builtin_nontemporal_load(reinterpret_cast<const typename HVec<V>::type*>(p + chunk * V));
    }
}
template <int V>
__device__ __forceinline__ void st_stream(_Float16* p, int64_t chunk, const typename HVec<V>::type& v)
{
    if constexpr (V == 1) {
        *reinterpret_cast<typename HVec<V>::type*>(p + chunk * V) = v;
    } else {
        __builtin_nontemporal_store(v, reinterpret_cast<typename HVec<V>::type*>(p + chunk * V));
    }
}

// Result stores with or without the hint.  Stores without it stay in the 256 MB memory-side cache: the pass that reads
// the result next finds it there, and a result that is overwritten soon (a pool of buffers, one call after another) may
// never reach memory.  That holds while result and reader fit the cache together, so results up to kCachedResultBytes
// are stored plainly.  us with the hint / plainly, a window quantiser and its inverse: 33 M 16-bit values (31 MiB of bytes,
// 63 MiB back) 38.5 / 36.0, 48 M 57.7 / 54.0, 64 M (bytes plain; values of 122 MiB hinted / plain) 66.0 / 69.8, 96 M (92 MiB
// of bytes, values hinted) 103.8 / 96.0, 128 M (122 MiB) 133 / 123; 16 M fp32 values 33.8 / 30.5, 64 M (61 MiB of bytes)
// 112.5 / 108.8, 96 M (92 MiB) 165 / 162.  A result that nothing reads: 16-bit bytes of 64 / 96 / 128 / 160 MiB 36.3 / 36.3,
// 51.9 / 53.9, 68.2 / 71.3, 84.5 / 87.8; values of 64 / 96 / 128 / 160 MiB 20.6 / 19.8, 29.2 / 29.9, 35.8 / 39.6, 44.0 / 48.3; a
// 268 MB int8 result 142 / 151.  Above 96 MiB what is gained with a reader is lost without one.
constexpr int64_t kCachedResultBytes = 96ll << 20;
// (The value is passed as a value: through a reference the compiler moves a load of quant_u8_kernel<16-bit type, 8> behind
// the store of the previous value, one load in flight per wavefront instead of eight, 1.24 ms for 0.48 at 1.0 G values.)
template <bool STREAM, typename T>
__device__ __forceinline__ void store_result(T* p, T v)
{
    if constexpr (STREAM) __builtin_nontemporal_store(v, p);
    else *p = v;
}

constexpr int kStreamThreads = 256;
constexpr int kStreamWaves = kStreamThreads / kWave;
constexpr int kMaxReduceChannels = 512;  // per-channel reductions: C/V <= 64 lane groups

// Default workgroup count of the persistent stream kernels.  Measured on MI355X with 256-thread
// workgroups at (1,64,350,350,128): 768 (three per CU, 3 wavefronts per SIMD) is fastest for the
// read-dominated and read+write fp16 streams, 512 for the pooling gather (whole multiples of the 256 CUs; 640 or 896 are measurably worse).
static inline int stream_blocks_default(int64_t work_items, int preferred = 768)
{
    int64_t b = ceil_div64(work_items, kStreamThreads);
    if (b > preferred) b = preferred;
    if (b < 1) b = 1;
    return (int)b;
}


// ---- launch shape of the flat stream kernels ------------------------------------------------------------
// A stream kernel walks its 16-byte chunks in steps of U chunks per thread (all U loads of a stream are issued
// before the first value is used).  With T = workgroups * threads, step k of a thread covers
//   interleaved (segment = 1): chunks k*U*T + u*T + b*threads + t          (a workgroup's chunks are T apart)
//   segments    (segment = U): chunks k*U*T + b*U*threads + u*threads + t  (a workgroup reads and writes one
//                                                                           contiguous run of U*threads chunks)
// for u < U; what is left after the last full step (< U*T chunks) is walked one chunk at a time.  Measured on
// MI355X with a plain copy of 2 GB: interleaved 256-thread workgroups reach 5.4-5.8 TB/s depending on the
// workgroup count (power-of-two counts such as 1024 fall to 4.4 TB/s: all accesses in flight then sit a
// power-of-two stride apart), 1024-thread workgroups on 128 KiB segments (U = 8) reach 6.0-6.3 TB/s whatever
// the count.  Both T and threads are multiples of the number of channel groups, so a thread keeps its group.
struct StreamShape {
    int blocks, threads, segment;  // segment: 1 = interleaved (U = 4), 4 or 8 = contiguous segments with that U
    int unroll() const { return segment == 8 ? 8 : 4; }
};
template <int U>
struct ChunkWalk {
    int64_t T, step, su, first, nfull, tail;
    __device__ __forceinline__ ChunkWalk(int64_t nchunks, bool segments)
    {
        const int64_t nthr = blockDim.x;
        T = (int64_t)gridDim.x * nthr;
        step = U * T;
        nfull = nchunks / step;
        su = segments ? nthr : T;
        first = (segments ? (int64_t)blockIdx.x * U * nthr : (int64_t)blockIdx.x * nthr) + threadIdx.x;
        tail = nfull * step + (int64_t)blockIdx.x * nthr + threadIdx.x;
    }
};
constexpr int kStreamMaxThreads = 1024;

// Sums of N values per lane over the lanes of a wavefront with the same lane % CG (CG <= 64 a power of two), pairs first at a
// distance of 32 lanes, then 16, ...  A step halves the values that a lane goes on with: it hands the other half of them to
// its partner, so N = 16 takes 8 + 4 + 2 + 1 exchanges, each step's in flight together, and one for every step after that.
// (A butterfly per value is N log2(64 / CG) exchanges one after the other, 96 at CG = 1: with fp32 values Stats of (1,8,64,64,32)
// 10.7 us, here 5.4, AddStats of (1,16,128,128,128) 40.4 and 36.1.)
// `store(base, v)`: called with the N >> steps values that the lane has, the first of them number `base`, by one lane each.
template <int N, int OFF = 32, class T, class Store>
__device__ __forceinline__ void wave_sums(T (&v)[N], int CG, int lane, int base, int spare, Store store)
{
    if constexpr (OFF > 0) {
        if (OFF >= CG) {  // (uniform)
            if constexpr (N > 1) {
                const bool up = (lane & OFF) != 0;
                T w[N / 2];
#pragma unroll
                for (int k = 0; k < N / 2; ++k) {
                    const T keep = up ? v[N / 2 + k] : v[k], give = up ? v[k] : v[N / 2 + k];
                    w[k] = keep + __shfl_xor(give, OFF, 64);
                }
                wave_sums<N / 2, OFF / 2>(w, CG, lane, base + (up ? N / 2 : 0), spare, store);
            } else {
                T w[1] = {v[0] + __shfl_xor(v[0], OFF, 64)};
                wave_sums<1, OFF / 2>(w, CG, lane, base, spare | OFF, store);  // both partners hold the sum
            }
            return;
        }
    }
    if ((lane & spare) == 0) {
#pragma unroll
        for (int k = 0; k < N; ++k) store(base + k, v[k]);
    }
}

typedef float fp32_pair_t __attribute__((ext_vector_type(2)));  // a sum rounded to fp32 and what the rounding left

// element `i` of a workspace of fp32 sums or, `pairs`, of fp32_pair_t
__device__ __forceinline__ void store_sum(float* ws, int64_t i, double sum, bool pairs)
{
    const float high = (float)sum;
    // (an infinite sum has no rest)
    if (pairs) reinterpret_cast<fp32_pair_t*>(ws)[i] = fp32_pair_t{high, __builtin_isfinite(high) ? (float)(sum - (double)high) : 0.0f};
    else ws[i] = high;
}

// Per-channel sums of a thread, then of its workgroup, in fp64.  A kernel adds the values of one step of its walk in fp32.  How
// many steps a thread takes, and how many workgroups there are, goes with the launch shape, which is chosen for its speed:
// with fp32 sums from step to step, over the lanes and in a workgroup's row, the error against 64 bits went with it.
// Relative errors, zero-mean values, all-fp32 sums / now: dscale of ApplyBNReLUBackward of (1,64,192,192,128) 316e-9 / 32e-9,
// dshift 69e-9 / 27e-9, mean of AddStats of (1,128,136,136,128) 43e-9 / 25e-9, of AvgPoolCeilStats of (1,64,61,63,63) 42e-9 /
// 25e-9.  Time: 0.3 us for the exchanges in fp64, 0.4 for the pairs, 1 to 2 % of the largest ApplyBNReLUBackward.
template <int V>
struct ChannelTotals {
    double tot[2 * V];
    __device__ __forceinline__ ChannelTotals()
    {
#pragma unroll
        for (int j = 0; j < 2 * V; ++j) tot[j] = 0.0;
    }
    __device__ __forceinline__ void take(float (&acc)[2][V])  // and clears acc
    {
#pragma unroll
        for (int j = 0; j < V; ++j) {
            tot[j] += (double)acc[0][j];
            tot[V + j] += (double)acc[1][j];
            acc[0][j] = acc[1][j] = 0.0f;
        }
    }
    // Adds the threads of the workgroup (up to 1024) that own the same channel group (thread t owns group t % CG, CG <= 64 a
    // power of two) and writes the workgroup's row of the workspace, [2][CG*V] sums as fp32 or, `pairs`, as fp32_pair_t.  The
    // wavefronts hand their sums over in rounds of four through LDS (`red`: 4*2*CG*V doubles); thread o keeps the running
    // sums of the outputs o, o + threads, ... (at most four of them: 2*512 / 256) and adds the rounds in a fixed order.
    __device__ __forceinline__ void write(int CG, double* red, float* ws, bool pairs)
    {
        const int t = threadIdx.x, lane = t % kWave, wave = t / kWave, nthr = blockDim.x, nwaves = nthr / kWave;
        const int cols = CG * V, nout = 2 * cols;
        constexpr int kMine = 4;
        double run[kMine];
#pragma unroll
        for (int m = 0; m < kMine; ++m) run[m] = 0.0;
        for (int r = 0; r < nwaves; r += 4) {
            if (wave >= r && wave < r + 4)
                wave_sums<2 * V>(tot, CG, lane, 0, 0, [&](int k, double v) {
                    red[((wave - r) * 2 + k / V) * cols + (lane & (CG - 1)) * V + k % V] = v;
                });
            __syncthreads();
#pragma unroll
            for (int m = 0; m < kMine; ++m) {
                const int o = t + m * nthr;
                if (o < nout) run[m] += ((red[o] + red[nout + o]) + (red[2 * nout + o] + red[3 * nout + o]));
            }
            if (r + 4 < nwaves) __syncthreads();
        }
#pragma unroll
        for (int m = 0; m < kMine; ++m) {
            const int o = t + m * nthr;
            if (o < nout) store_sum(ws, (int64_t)blockIdx.x * nout + o, run[m], pairs);
        }
    }
};

constexpr int kMaxDefaultBlocks = 4096;  // workspace queries with blocks = 0 size for this many partials
// `pairs` of ChannelTotals::write: where the launch shape is the library's own choice and the scratch memory has room for them (a
// workspace query with blocks = 0 does), unless the tensor is so small that its sums are short.
static inline bool sum_pairs(int blocks_asked, int blocks, int ncols, int64_t bytes, int64_t workspace_bytes)
{
    return blocks_asked <= 0 && workspace_bytes / (int64_t)sizeof(fp32_pair_t) >= (int64_t)blocks * ncols && bytes >= (8 << 20);
}

// Column sums in fp64 by a workgroup of 1024, in a fixed order: a slice of threads per row, N rows of a slice in flight at
// once, the slices of a wavefront combined in registers, the wavefronts' sums in LDS.  The buffer is small and was just
// written, so the trips to memory one after the other are what a sum costs: rows that do not exist are read from the last
// one and count as 0.0 instead of standing behind a condition or in a loop of their own (Stats of
// (1,32,48,48,48) 11.0 -> 10.0 us, DWConvWGRAD of it 15.0 -> 14.2, DWConvBackward of (1,16,40,40,40) 14.3 -> 13.7).
template <int N, class Row, class Add>
__device__ __forceinline__ void sum_slices(int nrows, int sl, int slices, Row row, Add add)
{
    for (int r0 = sl; r0 - sl < nrows; r0 += N * slices) {
        decltype(row(0)) v[N];
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = row(min(r0 + k * slices, nrows - 1));
#pragma unroll
        for (int k = 0; k < N; ++k) add(v[k], r0 + k * slices < nrows);
    }
}

// 32 columns (32 * blockIdx.x on) of a row-major fp32 buffer, 16-byte aligned, ncols a multiple of 32: returned by the
// threads below 32.  A workgroup takes a whole 128-byte line of every row, 16 bytes per lane.  (768 rows of 8192 columns:
// 6.9 us, 9.5 with 64 bytes of a row per workgroup and 4 bytes per lane.)
__device__ __forceinline__ double sum_lines(const float* __restrict__ ws, int nrows, int ncols, double (&part)[16][33])
{
    const int t = threadIdx.x, l = t % 8;
    const float4_t* col = reinterpret_cast<const float4_t*>(ws + blockIdx.x * 32) + l;
    const int64_t pitch = ncols / 4;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    auto row = [&](int r) { return col[r * pitch]; };
    auto add = [&](const float4_t& v, bool exists) {
#pragma unroll
        for (int k = 0; k < 4; ++k) s[k] += exists ? (double)v[k] : 0.0;
    };
    // (few rows: the wavefronts without one do not queue for the last one; ReLULinearBackward 32 -> 16 of 4000 / 9000 voxels 6.8 /
    // 7.0 us with sum_slices<2>, 6.2 / 6.6 so.  From 257 rows on the other way round: 64 -> 32 of 20000 8.9 / 9.1)
    if (nrows <= 256) {
        for (int r = t / 8; r < nrows; r += 128) add(row(r), true);
    } else if (nrows <= 512) {
        sum_slices<4>(nrows, t / 8, 128, row, add);
    } else {
        sum_slices<8>(nrows, t / 8, 128, row, add);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int off = 32; off >= 8; off >>= 1) s[k] += __shfl_xor(s[k], off, 64);
        if (t % kWave < 8) part[t / kWave][4 * l + k] = s[k];
    }
    __syncthreads();
    double v = 0.0;
    if (t < 32) {
#pragma unroll
        for (int w = 0; w < 16; ++w) v += part[w][t];
    }
    return v;
}

// 16 columns of any row-major buffer, column j (below ncols) per lane of 16: returned by the threads below 16.  T: float or
// fp32_pair_t.
__device__ __forceinline__ double wide(float v) { return (double)v; }
__device__ __forceinline__ double wide(fp32_pair_t v) { return (double)v[0] + (double)v[1]; }
template <class T>
__device__ __forceinline__ double sum_columns(const T* __restrict__ ws, int nrows, int64_t pitch, int j, int ncols,
                                              double (&part)[16][17])
{
    const int t = threadIdx.x;
    const T* col = ws + (j < ncols ? j : ncols - 1);
    double s = 0.0;
    auto row = [&](int r) { return col[r * pitch]; };
    auto add = [&](T v, bool exists) { s += exists ? wide(v) : 0.0; };
    if (nrows <= 256) sum_slices<4>(nrows, t / 16, 64, row, add);
    else sum_slices<8>(nrows, t / 16, 64, row, add);
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (t % kWave < 16) part[t / kWave][t % 16] = s;
    __syncthreads();
    double v = 0.0;
    if (t < 16) {
#pragma unroll
        for (int w = 0; w < 16; ++w) v += part[w][t];
    }
    return v;
}

// out[j] = scale * sum_r ws[r*ncols + j] for j < ncols, summed in fp64 in a fixed order;
// columns [0, split) go to out0, the rest to out1.  (Kernel lives in core.hip.)
void launch_reduce_rows(const float* ws, int nrows, int ncols, float* out0, float* out1, int split, double scale,
                        hipStream_t stream, bool pairs = false);
// the same for a multiple of 32 columns and scale 1, the results in out0 rounded to fp16
void launch_reduce_rows_f16(const float* ws, int nrows, int ncols, half_t* out0, float* out1, int split,
                            hipStream_t stream);
// result type of a gradient that a reduction kernel writes: fp32 or fp16
inline bool grad_dtype_ok(int dtype) { return dtype == KEROPS_DTYPE_F32 || dtype == KEROPS_DTYPE_F16; }

}  // namespace kerops
