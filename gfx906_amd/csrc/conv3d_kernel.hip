// Implicit-GEMM conv3d for AMD MI355X (gfx950 / CDNA4): fp16 NDHWC tensors,
// fp32 accumulation on matrix cores, fused fp16 bias + residual epilogue.
//
// Counterpart of the reference's VALU kernel (hip_conv/conv3d_kernel.hip:49-216,
// v_dot2_f32_f16 over a 128x64 tile), redesigned for CDNA4:
//
//  * GEMM view, transposed: O^T[k][m] = sum_i W[k][i] * X[m][i] with
//    m = ((n*Z + z)*P + p)*Q + q an output voxel, k an output channel and
//    i = ((t*R + r)*S + s)*C + c the reduction index, so that a packed
//    channels_last_3d weight row w[k] is contiguous in i and, with C % 8 == 0,
//    every aligned 8-element group of i lies in one (t, r, s) tap. With W as
//    the A operand of v_mfma_f32_16x16x32_f16, a lane's accumulator holds a
//    run of four consecutive output channels of one voxel: the
//    channels-innermost output, bias and residual move as 8-byte vectors.
//    (The card is power-limited under sustained matrix load; the 16x16x32
//    form costs less energy per FLOP than 32x32x16 and holds a higher clock:
//    +6 % on a VAE decoder layer.)
//  * Tiles of 64*CW channels x 32*NB*VW voxels x KB reduction elements (CW =
//    1, 2 or 4, VW = 2 or 4, NB = 1 to 4, KB = 32 or 64; nine configurations,
//    chosen per problem for how the tile count fills the CUs and how long the
//    reduction is), CW*VW waves of 64 x 32*NB (4 x 2NB MFMA blocks): with 4
//    waves two workgroups per CU whose barriers are independent, with 8 one
//    workgroup that loads fewer bytes per MFMA.
//    Both operand tiles go from HBM into LDS with buffer loads to LDS (no
//    VGPR staging); the input gather uses a per-lane offset (voxel base +
//    the offset of the lane's tap, advanced incrementally from k-tile to
//    k-tile), and lanes past M, K or the reduction length get an
//    out-of-range offset, so the load returns zeros. LDS rows are 2*KB bytes
//    (with KB = 64 each row is one whole 128-byte line of a weight row or of
//    a voxel's channels) with 16-byte units XOR-swizzled; a ring of two to
//    four stages keeps the loads of the next k-tiles in flight, k-tiles past
//    the end load zeros (so every wait count is static), and the barrier
//    waits for this wave's LDS reads only, not for loads in flight.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <algorithm>

#include "gfx906_amd_conv3d.h"
#include "scratch.h"

namespace {

using gfx906_amd::kScratchBytes;
using gfx906_amd::ScratchUse;

typedef _Float16 f16;
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define LDS_AS __attribute__((address_space(3)))

struct ConvArgs {
    const f16* x;
    const f16* w;
    const f16* bias;
    const f16* res;
    f16* out;
    int C, K, T, R, S, sd, sh, sw, Z, P, Q, M, KG;
    long long xsn, xsd, xsh, xsw, osn, osz, osp, osq, rsn, rsz, rsp, rsq;
    unsigned x_bytes, w_bytes;
    // Split reduction (nsplit > 1): split s takes reduction elements
    // [s*split_len, (s+1)*split_len) and writes its fp32 sums to
    // ws[s][m][k]; conv3d_reduce adds them up and runs the epilogue.
    int nsplit, split_len;
    float* ws;
};

constexpr int kMaxTaps = 1024;
constexpr long kMaxVoxels = (1L << 31) - 256;  // M
constexpr long kMaxBytes = 1L << 31;           // span of x or w
constexpr unsigned kOOB = 0xFFFFFFF0u;  // buffer offset past any range: loads zeros

// Per-configuration sizes: NB 32-voxel MFMA blocks per wave, CW waves along
// output channels x VW along voxels (64*CW channels x 32*NB*VW voxels per
// workgroup), NST stages in the LDS ring, KB reduction elements per k-tile
// (LDS rows of 2*KB bytes: 32 -> 64-byte rows, 64 -> 128-byte rows, so that
// each row of a tile is one whole 128-byte line of the weights or of a voxel).
template <int NB, int NST, int KB, int CW, int VW = 2>
struct ConvCfg {
    static constexpr int NW = VW * CW;              // waves
    static constexpr int NT = 64 * NW;              // threads
    static constexpr int BCH = 64 * CW;             // output channels per workgroup
    static constexpr int ROWB = 2 * KB;             // bytes per LDS row
    static constexpr int UNITS = ROWB / 16;         // 16-byte units per row
    static constexpr int RPB = 1024 / ROWB;         // rows per 1 KB load block
    static constexpr int BVX = 32 * NB * VW;        // output voxels per workgroup
    static constexpr int WTILE = BCH * ROWB;        // bytes of one W tile
    static constexpr int XTILE = BVX * ROWB;        // bytes of one X tile
    static constexpr int WJ = WTILE / 1024 / NW;    // W load blocks per wave per k-tile
    static constexpr int XBLK = XTILE / 1024;       // X load blocks per k-tile
    // X load blocks per wave per k-tile. When the waves do not divide the X
    // blocks, the waves past the last block issue a load of zeros into a
    // 1 KB pad after the X tile instead, so that every wave issues the same
    // number of loads and every wait count stays static.
    static constexpr int XJ = (XBLK + NW - 1) / NW;
    static constexpr int PAD = XJ * NW > XBLK ? 1024 : 0;
    static constexpr int STAGE = WTILE + XTILE + PAD;  // W tile, X tile, pad
    static constexpr int LOADS = WJ + XJ;
    static constexpr int OCC = NW == 4 ? 2 : 1;     // workgroups per CU
    static_assert(KB == 32 || KB == 64, "k-tile");
    static_assert(NW == 4 || NW == 8, "waves");
    static_assert(WJ * NW * 1024 == WTILE && XBLK * 1024 == XTILE, "whole load blocks");
    static_assert(NST * STAGE * OCC <= 160 * 1024, "LDS");
    static_assert(NST >= 2 && NST <= 4, "ring depth");
    static_assert((NST - 2) * LOADS < 16, "vmcnt immediate");
};

// Unit u of LDS row r sits in slot u ^ swz(r). 64-byte rows: four rows span
// the 64 banks and rows r, r+4 differ in swz; 128-byte rows: two rows span
// the banks and rows r, r+2, ..., r+14 differ in swz. Either way 16
// consecutive rows read at one unit cover 16 different bank groups.
template <int KB>
__host__ __device__ constexpr int swz(int r) { return KB == 32 ? (r >> 2) & 3 : (r >> 1) & 7; }

#if defined(__HIP_DEVICE_COMPILE__)
// Workgroup barrier for reusing an LDS stage: this wave's LDS reads are
// complete (lgkmcnt(0)), then s_barrier. Unlike __syncthreads() there is no
// release fence: that fence also waits for every outstanding load to LDS
// (vmcnt(0)), including the k-tiles meant to stay in flight. Each wave waits
// for its own part of the k-tile to be read (vmcnt(n)) before this. The
// memory clobber keeps the compiler from moving LDS accesses across it.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ f16x8 lds_read16(const char* base, int byte_off) {
    return *(const LDS_AS f16x8*)((const LDS_AS char*)base + byte_off);
}

// Output voxel m -> (n, z, p, q).
struct Voxel {
    int n, z, p, q;
};
__device__ __forceinline__ Voxel voxel(int m, int Z, int P, int Q) {
    Voxel v;
    v.q = m % Q;
    m /= Q;
    v.p = m % P;
    m /= P;
    v.z = m % Z;
    v.n = m / Z;
    return v;
}
#endif

// Tile (voxel tile * channel tiles + channel tile) of workgroup L of n.
// Workgroups go to the 8 XCDs round robin (L % 8), each XCD with its own L2;
// this map gives XCD x the x-th contiguous eighth of the tiles, in order, so
// that the channel tiles of one voxel tile, and neighbouring voxel tiles
// (whose input windows overlap), share one L2.
__device__ __forceinline__ int tile_of(int L, int n) {
    const int xcd = L & 7, pos = L >> 3, base = n >> 3, extra = n & 7;
    return (xcd < extra ? xcd * (base + 1) : extra * (base + 1) + (xcd - extra) * base) + pos;
}

#if defined(__HIP_DEVICE_COMPILE__)
// One workgroup of conv3d_mfma (SPLIT: of conv3d_part). SMALLC: C < KB, so
// that one k-tile can cross several taps.
template <int NB, int NST, int KB, int CW, int VW, bool SMALLC, bool SPLIT>
__device__ __forceinline__ void conv_tile(const ConvArgs a) {
    using Cf = ConvCfg<NB, NST, KB, CW, VW>;
    constexpr int STAGE = Cf::STAGE, LOADS = Cf::LOADS, ROWB = Cf::ROWB, UNITS = Cf::UNITS;
    constexpr int RPB = Cf::RPB, WJ = Cf::WJ, XJ = Cf::XJ, NW = Cf::NW;
    // The ring's stages are separate arrays, so that the compiler can tell
    // their accesses apart: a read of one stage never waits for the loads
    // into another.
    __shared__ __attribute__((aligned(1024))) char st0[STAGE];
    __shared__ __attribute__((aligned(1024))) char st1[STAGE];
    __shared__ __attribute__((aligned(1024))) char st2[NST > 2 ? STAGE : 16];
    __shared__ __attribute__((aligned(1024))) char st3[NST > 3 ? STAGE : 16];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Work item: split-major, so that with a split reduction an XCD's
    // workgroups share the weights and taps of one or two ranges.
    int m0, k0, split = 0;
    {
        const int nct = (a.K + Cf::BCH - 1) / Cf::BCH;
        int t = tile_of(blockIdx.x, gridDim.x);
        if constexpr (SPLIT) {
            const int ntiles = (int)gridDim.x / a.nsplit;
            split = t / ntiles;
            t -= split * ntiles;
        }
        const int vt = t / nct;
        m0 = vt * Cf::BVX;
        k0 = (t - vt * nct) * Cf::BCH;
    }
    // This workgroup's reduction range.
    const int i_beg = SPLIT ? split * a.split_len : 0;
    const int i_end = SPLIT ? min(a.KG, i_beg + a.split_len) : a.KG;

    // Load roles. LDS block b (1 KB) holds rows RPB*b..RPB*b+RPB-1 of a tile;
    // lane l writes row RPB*b + l/UNITS, slot l%UNITS, so it fetches unit
    // u = (l%UNITS) ^ swz(row). For the lane's blocks (W blocks wave + NW*j,
    // j < WJ; X blocks wave + NW*j, j < XJ) swz(row) does not depend on j, so
    // u and the tap of the lane's reduction group are the same in all of them.
    const int rsub = lane / UNITS;
    const int u = (lane % UNITS) ^ swz<KB>(RPB * wave + rsub);
    unsigned wo[WJ];  // bytes into w (unused, and possibly wrapped, for rows past K)
    bool wv[WJ];
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
        const int k = k0 + RPB * (wave + NW * j) + rsub;
        wv[j] = k < a.K;
        wo[j] = ((unsigned)k * (unsigned)a.KG + 8u * (unsigned)u) * 2u;
    }
    int xo[XJ];
    bool xv[XJ];
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
        const int m = m0 + RPB * (wave + NW * j) + rsub;
        xv[j] = m < a.M && wave + NW * j < Cf::XBLK;
        const Voxel v = voxel(m, a.Z, a.P, a.Q);
        xo[j] = (int)(v.n * a.xsn + (long long)v.z * a.sd * a.xsd +
                      (long long)v.p * a.sh * a.xsh + (long long)v.q * a.sw * a.xsw);
    }
    const __amdgpu_buffer_rsrc_t rw =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.w, 0, (int)a.w_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, (int)a.x_bytes, 0x00020000);

    // The lane's reduction group of the next k-tile to issue: reduction index
    // gi = i0 + 8u lies in tap (t, r, s) at channel cc, and the tap starts
    // toff elements into a window (toff = t*xsd + r*xsh + s*xsw). The tap is
    // advanced incrementally, so the loop reads no tap table.
    int gi = i_beg + 8 * u;
    int cc, ts, tr, toff;
    {
        const int tp = gi / a.C;
        cc = gi - tp * a.C;
        ts = tp % a.S;
        tr = (tp / a.S) % a.R;
        const int tt = tp / (a.S * a.R);
        toff = (int)(tt * a.xsd + tr * a.xsh + ts * a.xsw);
    }
    // Per k-tile the group moves KB = tstep*C + cstep elements on: whole taps
    // (C < KB only), then cstep channels with at most one more tap.
    const int tstep = SMALLC ? KB / a.C : 0;
    const int cstep = KB - tstep * a.C;
    const int dr = (int)(a.xsh - a.S * a.xsw), dt = (int)(a.xsd - a.R * a.xsh);
    // Next tap where `go` holds: s, then r, then t.
    auto next_tap = [&](bool go) __attribute__((always_inline)) {
        ts += go ? 1 : 0;
        toff += go ? (int)a.xsw : 0;
        const bool ws = ts == a.S;
        ts = ws ? 0 : ts;
        tr += ws ? 1 : 0;
        toff += ws ? dr : 0;
        const bool wr = tr == a.R;
        tr = wr ? 0 : tr;
        toff += wr ? dt : 0;
    };

    // Loads of the next k-tile (reduction indices i0 .. i0+KB-1) into an LDS
    // stage, then the lane's group moves on by KB.
    int i0 = i_beg;
    auto issue = [&](char* dst) __attribute__((always_inline)) {
        const bool kin = gi < i_end;
#pragma unroll
        for (int j = 0; j < WJ; ++j) {
            const unsigned ow = (wv[j] && kin) ? wo[j] + 2u * (unsigned)i0 : kOOB;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rw, (LDS_AS void*)(dst + (wave + NW * j) * 1024), 16, (int)ow, 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < XJ; ++j) {
            const unsigned ox = (xv[j] && kin) ? (unsigned)(2 * (xo[j] + toff + cc)) : kOOB;
            const int blk = wave + NW * j;  // past the X tile: zeros into the pad
            char* xdst = dst + Cf::WTILE + (blk < Cf::XBLK ? blk * 1024 : Cf::XTILE);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (LDS_AS void*)xdst, 16, (int)ox, 0, 0, 0);
        }
        i0 += KB;
        gi += KB;
        if (SMALLC) {  // tstep <= KB / 8 for C >= 8
#pragma unroll
            for (int i = 0; i < KB / 8; ++i) next_tap(i < tstep);
        }
        cc += cstep;
        const bool wrap = cc >= a.C;
        cc -= wrap ? a.C : 0;
        next_tap(wrap);
    };

    // MFMA operand addresses (v_mfma_f32_16x16x32_f16): lane l reads row
    // (16-row block base + l%16), unit 4*ks + l/16 (32 reduction elements per
    // k-step).
    constexpr int KS32 = KB / 32;
    const int g = lane >> 4, r16 = lane & 15;
    const int wch = wave % CW, wvx = wave / CW;  // channel quarter/half, voxel half
    int aaddr[4][KS32], baddr[2 * NB][KS32];
#pragma unroll
    for (int ks = 0; ks < KS32; ++ks) {
#pragma unroll
        for (int bl = 0; bl < 4; ++bl) {
            const int ra = wch * 64 + bl * 16 + r16;
            aaddr[bl][ks] = ra * ROWB + (((4 * ks + g) ^ swz<KB>(ra)) * 16);
        }
#pragma unroll
        for (int bl = 0; bl < 2 * NB; ++bl) {
            const int rb = wvx * 32 * NB + bl * 16 + r16;
            baddr[bl][ks] = Cf::WTILE + rb * ROWB + (((4 * ks + g) ^ swz<KB>(rb)) * 16);
        }
    }

    f32x4 acc[4][2 * NB];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
        for (int vb = 0; vb < 2 * NB; ++vb) acc[cb][vb] = f32x4{};

    // One k-tile from stage cur, after issuing the loads of the k-tile NST-1
    // ahead into fill (the stage of the k-tile before this one).
    auto step = [&](char* __restrict__ fill, const char* __restrict__ cur)
        __attribute__((always_inline)) {
        // vmcnt(NST-2 k-tiles of loads): this wave's part of the k-tile in cur
        // landed.
        __builtin_amdgcn_s_waitcnt(0x0F70 | ((NST - 2) * LOADS));
        lds_barrier();    // every wave's; the k-tile in fill was consumed
        issue(fill);
        f16x8 af[KS32][4], bf[KS32][2 * NB];
#pragma unroll
        for (int ks = 0; ks < KS32; ++ks) {
#pragma unroll
            for (int bl = 0; bl < 4; ++bl) af[ks][bl] = lds_read16(cur, aaddr[bl][ks]);
#pragma unroll
            for (int bl = 0; bl < 2 * NB; ++bl) bf[ks][bl] = lds_read16(cur, baddr[bl][ks]);
        }
#pragma unroll
        for (int ks = 0; ks < KS32; ++ks)
#pragma unroll
            for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                for (int vb = 0; vb < 2 * NB; ++vb)
                    acc[cb][vb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[ks][cb], bf[ks][vb],
                                                                         acc[cb][vb], 0, 0, 0);
        // With the small-C tap walk, a k-tile's reads hoisted above the
        // previous k-tile's MFMAs push the wave past 256 VGPRs (spills).
        if constexpr (SMALLC) __builtin_amdgcn_sched_barrier(0);
    };
    // k-tile t sits in stage t % NST. The loop runs whole groups of NST
    // k-tiles: k-tiles past the end load zeros and add nothing.
    const int nkt = (i_end - i_beg + KB - 1) / KB;
    issue(st0);
    if constexpr (NST == 2) {
        for (int kt = 0; kt < nkt; kt += 2) {
            step(st1, st0);
            step(st0, st1);
        }
    } else if constexpr (NST == 4) {
        issue(st1);
        issue(st2);
        for (int kt = 0; kt < nkt; kt += 4) {
            step(st3, st0);
            step(st0, st1);
            step(st1, st2);
            step(st2, st3);
        }
    } else {
        issue(st1);
        for (int kt = 0; kt < nkt; kt += 3) {
            step(st2, st0);
            step(st0, st1);
            step(st1, st2);
        }
    }
    // The zero loads past the last k-tile must land before the workgroup's
    // LDS is released.
    __builtin_amdgcn_s_waitcnt(0x0F70);

    if constexpr (SPLIT) {  // this range's sums, in the accumulators' order
#pragma unroll
        for (int vb = 0; vb < 2 * NB; ++vb) {
            const int m = m0 + wvx * 32 * NB + vb * 16 + r16;
            if (m >= a.M) continue;
            float* row = a.ws + ((long long)split * a.M + m) * a.K;
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) {
                const int ch = k0 + wch * 64 + cb * 16 + 4 * g;
                if (ch < a.K) *(f32x4*)(row + ch) = acc[cb][vb];
            }
        }
        return;
    }
    // Epilogue: accumulator row 4g + r (an output channel), column l%16 (an
    // output voxel); one run of four channels per lane, voxel and block.
#pragma unroll
    for (int vb = 0; vb < 2 * NB; ++vb) {
        const int m = m0 + wvx * 32 * NB + vb * 16 + r16;
        if (m >= a.M) continue;
        const Voxel v = voxel(m, a.Z, a.P, a.Q);
        const long long oo = v.n * a.osn + v.z * a.osz + v.p * a.osp + v.q * a.osq;
        const long long ro = v.n * a.rsn + v.z * a.rsz + v.p * a.rsp + v.q * a.rsq;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const int ch = k0 + wch * 64 + cb * 16 + 4 * g;
            if (ch >= a.K) continue;
            f32x4 val = acc[cb][vb];
            if (a.bias) val += __builtin_convertvector(*(const f16x4*)(a.bias + ch), f32x4);
            if (a.res) val += __builtin_convertvector(*(const f16x4*)(a.res + ro + ch), f32x4);
            *(f16x4*)(a.out + oo + ch) = __builtin_convertvector(val, f16x4);
        }
    }
}
#endif

// grid: ceil(M / (64*NB)) * ceil(K / (64*CW)) workgroups (1-D, see tile_of);
// block: 128*CW threads. The second launch bound is HIP's minimum waves per
// SIMD (amdgpu_waves_per_eu): OCC workgroups of 2*CW waves over the CU's four
// SIMDs.
template <int NB, int NST, int KB, int CW, bool SMALLC>
__global__ void __launch_bounds__((ConvCfg<NB, NST, KB, CW>::NT),
                                  (ConvCfg<NB, NST, KB, CW>::OCC * ConvCfg<NB, NST, KB, CW>::NW / 4))
    conv3d_mfma(const ConvArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    conv_tile<NB, NST, KB, CW, 2, SMALLC, false>(a);
#endif
}

// Any number of voxel waves and, with SPLIT, the reduction split in a.nsplit
// ranges: nsplit times as many workgroups, split-major. (Kernels of their own:
// a range's bounds and second epilogue cost the unsplit form 1 %.)
template <int NB, int NST, int KB, int CW, int VW, bool SMALLC, bool SPLIT>
__global__ void __launch_bounds__((ConvCfg<NB, NST, KB, CW, VW>::NT),
                                  (ConvCfg<NB, NST, KB, CW, VW>::OCC *
                                   ConvCfg<NB, NST, KB, CW, VW>::NW / 4))
    conv3d_part(const ConvArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    conv_tile<NB, NST, KB, CW, VW, SMALLC, SPLIT>(a);
#endif
}

// Sum of a split reduction's partial results in split order, then the epilogue
// of conv3d_mfma. One thread per voxel and 4 channels; the loads of
// kRedBatch splits go out together (the partial results of a problem small
// enough to be split mostly come from the caches, so latency, not bandwidth,
// would bound a loop that waited for each split in turn).
constexpr int kRedBatch = 4;
__global__ void __launch_bounds__(256) conv3d_reduce(const ConvArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    const int kq = a.K / 4;
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long long)a.M * kq) return;
    const int m = (int)(idx / kq), ch = (int)(idx - (long long)m * kq) * 4;
    const float* part = a.ws + (long long)m * a.K + ch;
    const long long step = (long long)a.M * a.K;
    f32x4 val = {};
    for (int s0 = 0; s0 < a.nsplit; s0 += kRedBatch) {
        f32x4 p[kRedBatch];
#pragma unroll
        for (int u = 0; u < kRedBatch; ++u)
            if (s0 + u < a.nsplit) p[u] = *(const f32x4*)(part + (s0 + u) * step);
#pragma unroll
        for (int u = 0; u < kRedBatch; ++u)
            if (s0 + u < a.nsplit) val += p[u];
    }
    const Voxel v = voxel(m, a.Z, a.P, a.Q);
    if (a.bias) val += __builtin_convertvector(*(const f16x4*)(a.bias + ch), f32x4);
    if (a.res)
        val += __builtin_convertvector(
            *(const f16x4*)(a.res + v.n * a.rsn + v.z * a.rsz + v.p * a.rsp + v.q * a.rsq + ch),
            f32x4);
    *(f16x4*)(a.out + v.n * a.osn + v.z * a.osz + v.p * a.osp + v.q * a.osq + ch) =
        __builtin_convertvector(val, f16x4);
#endif
}

// Launches configuration (NB, NST, KB, CW, VW) over the whole problem.
template <int NB, int NST, int KB, int CW, int VW, bool SMALLC>
void launch_c(const ConvArgs& a, hipStream_t stream) {
    using Cf = ConvCfg<NB, NST, KB, CW, VW>;
    const unsigned tiles = (unsigned)((a.M + Cf::BVX - 1) / Cf::BVX) *
                           (unsigned)((a.K + Cf::BCH - 1) / Cf::BCH) * (unsigned)a.nsplit;
    const dim3 grid(tiles), block(Cf::NT);
    if (a.nsplit > 1)
        hipLaunchKernelGGL((conv3d_part<NB, NST, KB, CW, VW, SMALLC, true>), grid, block, 0, stream,
                           a);
    else if constexpr (VW == 2)
        hipLaunchKernelGGL((conv3d_mfma<NB, NST, KB, CW, SMALLC>), grid, block, 0, stream, a);
    else
        hipLaunchKernelGGL((conv3d_part<NB, NST, KB, CW, VW, SMALLC, false>), grid, block, 0,
                           stream, a);
}
template <int NB, int NST, int KB, int CW, int VW = 2>
void launch_cfg(const ConvArgs& a, hipStream_t stream) {
    if (a.C < KB)
        launch_c<NB, NST, KB, CW, VW, true>(a, stream);
    else
        launch_c<NB, NST, KB, CW, VW, false>(a, stream);
}

thread_local char g_err[256];

void set_err(const char* msg) {
    int i = 0;
    for (; msg[i] && i < 255; ++i) g_err[i] = msg[i];
    g_err[i] = 0;
}

int fail(const char* msg) {
    set_err(msg);
    return 1;
}

bool mult8(long v) { return v >= 0 && v % 8 == 0; }

// The kernel configurations: voxels / 64, KB, channels per workgroup (64*CW),
// workgroups per CU, ring stages; the time in us of a 64-voxel x 256-channel
// piece of a tile (`per_kg` for a reduction of 13824 elements, `fixed` for
// start-up and epilogue); how much of it a workgroup that shares its CU takes
// longer than one alone, and an odd last one; the factor on per_kg where C < 64
// (taps change within a k-tile); launcher. Fitted on MI355X, see plan_conv. The
// last two have four waves along the voxels: 256 voxels x 128 channels in one
// workgroup of eight waves load a quarter less per output than two workgroups of
// 128 x 128 (a strided 128 -> 128 layer of 65,536 voxels 69 -> 64 us, stride 1
// 66 -> 58), 128 x 64 wastes less on 64 and 192 channels (64 -> 64 of 98,304
// voxels 49 -> 35 us) and makes more, shorter workgroups of small problems (512
// -> 512 of 256 voxels 22 -> 16 us).
struct ConvKernel {
    int nb, kb, bch, occ, nst;
    double per_kg, fixed, shared, odd, small_c;
    void (*launch)(const ConvArgs&, hipStream_t);
};
const ConvKernel kKernels[] = {
    {4, 32, 128, 2, 3, 85.0, 3.6, 0.88, 0.15, 0.88, launch_cfg<4, 3, 32, 2>},
    {3, 64, 128, 2, 2, 88.0, 3.8, 0.40, 0.32, 0.85, launch_cfg<3, 2, 64, 2>},
    {2, 64, 128, 2, 2, 93.0, 4.7, 0.18, 0.63, 0.85, launch_cfg<2, 2, 64, 2>},
    {4, 32, 256, 1, 4, 77.0, 3.6, 0.0, 0.0, 0.92, launch_cfg<4, 4, 32, 4>},
    {3, 64, 256, 1, 2, 86.0, 3.4, 0.0, 0.0, 0.92, launch_cfg<3, 2, 64, 4>},
    {2, 64, 256, 1, 3, 79.0, 3.8, 0.0, 0.0, 1.22, launch_cfg<2, 3, 64, 4>},
    {3, 32, 256, 1, 4, 86.0, 3.6, 0.0, 0.0, 0.85, launch_cfg<3, 4, 32, 4>},
    {4, 64, 128, 1, 3, 79.0, 5.0, 0.0, 0.0, 1.09, launch_cfg<2, 3, 64, 2, 4>},
    {2, 64, 64, 2, 3, 112.0, 6.7, 0.74, 0.05, 1.24, launch_cfg<1, 3, 64, 1, 4>},
};
constexpr int kNumKernels = sizeof(kKernels) / sizeof(kKernels[0]);

int find_kernel(int nb, int kb, int bch) {
    for (int i = 0; i < kNumKernels; ++i)
        if (kKernels[i].nb == nb && kKernels[i].kb == kb && kKernels[i].bch == bch) return i;
    return -1;
}

// Kernel configuration and split of the reduction for an M x K problem with
// reduction length KG: the pair with the least estimated time. Wider tiles
// load fewer bytes per MFMA (the loads into LDS, not the matrix cores, bound
// these kernels); narrower ones fill the CUs better when the tile count is
// small or just past a multiple of the workgroup slots. 64-wide k-tiles fetch
// whole 128-byte lines, 32-wide ones half lines but leave room for a deeper
// ring. A problem with fewer tiles than slots splits the reduction into
// nsplit ranges of whole 64-element units: without it a 32x32x2-voxel layer of
// 512 channels (64 tiles of 216 serial k-tiles) left three quarters of the
// CUs idle and took 183 us; in 8 ranges it takes 42.
// Estimate: tile size x (R x per_kg x range / 13824 + R' x fixed), the range in
// whole groups of ring stages, R the workgroups on the busiest CU in units of one
// workgroup's time (for two per CU: halves of a pair's time, one workgroup alone
// taking 2 - `shared` halves and an odd last one 1 + `odd`; of the fixed part,
// which is latency, one alone takes 2 - kFixedShared), plus for a split the
// reduce kernel: a launch, a little per range (its loads go out four ranges at a
// time) and the partial sums' traffic. Fitted to 900 layers on MI355X (1x1x1 to
// 3x3x3 windows, 8 to 512 channels, 200 to 200,000 voxels) over every
// configuration and 1 to 48 ranges. On 360 others the chosen pair is 0.6 % behind
// the fastest one on average, and 2 of them are more than 3 % (up to 11 %) slower
// than with the seven 128- and 256-channel configurations and no split, as they
// were chosen before the last two configurations and the splits came. A fit to 24
// layers, hardly any with C < 64 or a reduction under 500, was 1.6 % behind and
// slower there on one layer in 20, up to 22 % (384 -> 512 of 8250 voxels, 1x1x1
// window: 17.3 us, 14.4 with what is chosen now).
// For tests, read on every call: GFX906_AMD_CONV_CFG = "<NB>x<KB>" (128
// channels) or "<NB>x<KB>x<channels>" (a row of kKernels) fixes the
// configuration, unsplit unless GFX906_AMD_CONV_NSPLIT = n asks for n ranges
// (as many as there are units at most, fewer where n does not divide them
// into non-empty ranges, none where the partial sums exceed ws_cap).
constexpr int kSplitUnit = 64;     // reduction elements
constexpr int kSplitMinUnits = 4;  // shortest range worth a workgroup
constexpr int kSplitMax = 64;
// A split has to be this much better than none: CUs left idle let the others
// hold a higher clock (512 -> 512 of 17,812 voxels, 186 workgroups unsplit: 250
// us, and 274 in two ranges that the estimate has 7 % ahead).
constexpr double kSplitMargin = 1.12;
constexpr double kRedLaunch = 1.33, kRedPerSplit = 0.09, kRedPerByte = 0.17e-6;  // us
constexpr double kFixedShared = 0.57;
constexpr int kSmallC = 64;
constexpr double kSmallCFixed = 1.2;  // factor on `fixed` where C < 64
struct ConvPlan {
    int cfg, nsplit, split_len;
};

size_t conv_ws_bytes(const ConvPlan& p, long M, int K) {
    return p.nsplit <= 1 ? 0 : (size_t)p.nsplit * M * K * 4;
}

unsigned conv_cus() {
    static const unsigned ncu = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            n <= 0)
            n = 256;
        return (unsigned)n;
    }();
    return ncu;
}

// Tiles of a configuration (held to 2^24, an output past the device's memory, so
// that 32 bits count the ranges too).
unsigned conv_tiles(const ConvKernel& c, long M, int K) {
    return (unsigned)std::min((M + 64 * c.nb - 1) / (64 * c.nb) * (((long)K + c.bch - 1) / c.bch),
                              1L << 24);
}

// Estimated time of `wgs` workgroups over `range` reduction elements each.
double conv_cost(const ConvKernel& c, unsigned wgs, unsigned range, unsigned ncu, bool small_c) {
    const unsigned group = (unsigned)(c.nst * c.kb);
    const double kgu = (double)((range + group - 1) / group * group) / 13824.0;
    const unsigned n = (wgs + ncu - 1) / ncu;
    double r = n, r_fixed = n;  // workgroups on the busiest CU
    if (c.occ == 2 && n == 1) {
        r = 2.0 - c.shared;
        r_fixed = 2.0 - kFixedShared;
    } else if (c.occ == 2 && (n & 1)) {
        r += c.odd;
    }
    return c.nb * c.bch / 256.0 * (r * c.per_kg * (small_c ? c.small_c : 1.0) * kgu +
                                   r_fixed * c.fixed * (small_c ? kSmallCFixed : 1.0));
}

// The configuration that GFX906_AMD_CONV_CFG names, or -1.
int forced_kernel() {
    const char* e = getenv("GFX906_AMD_CONV_CFG");
    int nb = 0, kb = 0, bch = 128;
    return e && sscanf(e, "%dx%dx%d", &nb, &kb, &bch) >= 2 ? find_kernel(nb, kb, bch) : -1;
}

ConvPlan plan_conv(long M, int K, long KG, size_t ws_cap) {
    const unsigned ncu = conv_cus();
    const int only = forced_kernel();
    const long units = (KG + kSplitUnit - 1) / kSplitUnit;
    unsigned tiles1[kNumKernels], fewest = ~0u;  // tiles of each configuration, unsplit
    for (int i = 0; i < kNumKernels; ++i) {
        tiles1[i] = conv_tiles(kKernels[i], M, K);
        fewest = std::min(fewest, tiles1[i]);
    }
    // More than four rounds of workgroups gain nothing (and the search costs
    // host time on every call).
    long ns_lo = 1, ns_hi = only >= 0 ? 1
                                      : std::min({units / kSplitMinUnits, (long)kSplitMax,
                                                  (long)(4 * ncu / fewest)});
    if (const char* e = getenv("GFX906_AMD_CONV_NSPLIT")) {
        const long n = atol(e);
        if (n >= 1) ns_lo = ns_hi = std::min(n, units);
    }
    ConvPlan best{only >= 0 ? only : 0, 1, (int)KG};
    double best_cost = 1e300;
    for (long ns = ns_lo; ns <= std::max(ns_lo, ns_hi); ++ns) {
        const long per = (units + ns - 1) / ns;
        const ConvPlan p{0, (int)((units + per - 1) / per), (int)(per * kSplitUnit)};
        if (ns > ns_lo && p.nsplit != ns) continue;  // the same ranges as a smaller count
        if (conv_ws_bytes(p, M, K) > ws_cap) break;
        const unsigned range = (unsigned)std::min<long>(KG, p.split_len);
        const double red = p.nsplit > 1 ? kRedLaunch + kRedPerSplit * p.nsplit +
                                              kRedPerByte * (double)conv_ws_bytes(p, M, K)
                                        : 0.0;
        for (int i = 0; i < kNumKernels; ++i) {
            if (only >= 0 && i != only) continue;
            double cost =
                conv_cost(kKernels[i], tiles1[i] * (unsigned)p.nsplit, range, ncu, false) + red;
            if (p.nsplit > 1) cost *= kSplitMargin;
            if (cost < best_cost) {
                best_cost = cost;
                best = p;
                best.cfg = i;
            }
        }
    }
    return best;
}

// The plan's configuration where C < 64, for the same ranges (the workspace, and
// with it the ranges, is planned without C).
int small_c_kernel(const ConvPlan& p, long M, int K, long KG) {
    if (forced_kernel() >= 0) return p.cfg;
    const unsigned ncu = conv_cus(), range = (unsigned)std::min<long>(KG, p.split_len);
    int best = p.cfg;
    double best_cost = 1e300;
    for (int i = 0; i < kNumKernels; ++i) {
        const double cost = conv_cost(kKernels[i], conv_tiles(kKernels[i], M, K) * (unsigned)p.nsplit,
                                      range, ncu, true);
        if (cost < best_cost) {
            best_cost = cost;
            best = i;
        }
    }
    return best;
}

}  // namespace

extern "C" const char* conv3d_last_error(void) { return g_err[0] ? g_err : nullptr; }

namespace {

// conv3d_fwd and launch_conv3d (use_scratch: a split reduction's partial
// results go to the static scratch) and conv3d_fwd_split (caller workspace).
int conv3d_impl(const void* x, const void* w, const void* bias, const void* res, void* out, int nB,
                int D, int H, int W, int C, int K, int T, int R, int S, int sd, int sh, int sw,
                int Z, int P, int Q, long M, long xsn, long xsd, long xsh, long xsw, long osn,
                long osz, long osp, long osq, long rsn, long rsz, long rsp, long rsq,
                hipStream_t stream, void* workspace, size_t workspace_bytes, bool use_scratch) {
    g_err[0] = 0;
    if (nB <= 0 || D <= 0 || H <= 0 || W <= 0 || C <= 0 || K <= 0 || T <= 0 || R <= 0 || S <= 0)
        return fail("conv3d: sizes must be positive");
    if (sd <= 0 || sh <= 0 || sw <= 0) return fail("conv3d: strides must be positive");
    if (C % 8 || K % 8) return fail("conv3d: C and K must be multiples of 8");
    if (D < T || H < R || W < S || Z != (D - T) / sd + 1 || P != (H - R) / sh + 1 ||
        Q != (W - S) / sw + 1)
        return fail("conv3d: output size does not match a VALID convolution");
    if (M != (long)nB * Z * P * Q || M >= kMaxVoxels)
        return fail("conv3d: M must be nB*Z*P*Q < 2^31 - 256");
    if ((long)T * R * S > kMaxTaps) return fail("conv3d: more than 1024 taps");
    if (!x || !w || !out) return fail("conv3d: null pointer");
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)res) % 16 ||
        (uintptr_t)bias % 8)
        return fail("conv3d: x, w, out, res must be 16-byte and bias 8-byte aligned");
    const long strides[12] = {xsn, xsd, xsh, xsw, osn, osz, osp, osq, rsn, rsz, rsp, rsq};
    for (long s : strides)
        if (!mult8(s)) return fail("conv3d: strides must be non-negative multiples of 8");
    const long KG = (long)C * T * R * S;
    const long x_span = ((nB - 1) * xsn + (D - 1) * xsd + (H - 1) * xsh + (W - 1) * xsw + C) * 2;
    const long w_span = (long)K * KG * 2;
    if (x_span >= kMaxBytes || w_span >= kMaxBytes)
        return fail("conv3d: x or w spans 2^31 bytes or more");
    ConvArgs a;
    a.x = (const f16*)x;
    a.w = (const f16*)w;
    a.bias = (const f16*)bias;
    a.res = (const f16*)res;
    a.out = (f16*)out;
    a.C = C;
    a.K = K;
    a.T = T;
    a.R = R;
    a.S = S;
    a.sd = sd;
    a.sh = sh;
    a.sw = sw;
    a.Z = Z;
    a.P = P;
    a.Q = Q;
    a.M = (int)M;
    a.KG = (int)KG;
    a.xsn = xsn;
    a.xsd = xsd;
    a.xsh = xsh;
    a.xsw = xsw;
    a.osn = osn;
    a.osz = osz;
    a.osp = osp;
    a.osq = osq;
    a.rsn = rsn;
    a.rsz = rsz;
    a.rsp = rsp;
    a.rsq = rsq;
    a.x_bytes = (unsigned)x_span;
    a.w_bytes = (unsigned)w_span;
    ConvPlan p = plan_conv(M, K, KG, kScratchBytes);
    ScratchUse scratch;
    if (p.nsplit > 1 && use_scratch) {
        // A captured call takes no scratch (its replays could run beside other
        // calls that use it) and runs unsplit.
        const size_t need = conv_ws_bytes(p, M, K);
        const ScratchUse::Status st = scratch.acquire(stream, need, false);
        if (st == ScratchUse::kFailed) {
            set_err(scratch.error);
            return 2;
        }
        if (st == ScratchUse::kUnavailable) p = plan_conv(M, K, KG, 0);
        workspace = scratch.ptr;
        workspace_bytes = need;
    }
    if (p.nsplit > 1 && (!workspace || workspace_bytes < conv_ws_bytes(p, M, K) ||
                         (uintptr_t)workspace % 16))
        return fail("conv3d: workspace missing, misaligned or smaller than "
                    "conv3d_workspace_bytes()");
    a.nsplit = p.nsplit;
    a.split_len = p.split_len;
    a.ws = (float*)workspace;
    if (C < kSmallC) p.cfg = small_c_kernel(p, M, K, KG);
    kKernels[p.cfg].launch(a, stream);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && p.nsplit > 1) {
        const long threads = M * (K / 4);
        hipLaunchKernelGGL(conv3d_reduce, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                           stream, a);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = scratch.release();
    if (e != hipSuccess) {
        set_err(hipGetErrorString(e));
        return 2;
    }
    return 0;
}

}  // namespace

extern "C" int conv3d_fwd(const void* x, const void* w, const void* bias, const void* res,
                          void* out, int nB, int D, int H, int W, int C, int K, int T, int R, int S,
                          int sd, int sh, int sw, int Z, int P, int Q, long M, long xsn, long xsd,
                          long xsh, long xsw, long osn, long osz, long osp, long osq, long rsn,
                          long rsz, long rsp, long rsq, hipStream_t stream) {
    return conv3d_impl(x, w, bias, res, out, nB, D, H, W, C, K, T, R, S, sd, sh, sw, Z, P, Q, M,
                       xsn, xsd, xsh, xsw, osn, osz, osp, osq, rsn, rsz, rsp, rsq, stream, nullptr,
                       0, true);
}

extern "C" size_t conv3d_workspace_bytes(long M, int K, long KG) {
    // Sizes that conv3d_fwd_split() refuses need none.
    if (M <= 0 || K <= 0 || KG <= 0 || M >= kMaxVoxels || KG >= kMaxBytes ||
        (long)K * KG * 2 >= kMaxBytes)
        return 0;
    return conv_ws_bytes(plan_conv(M, K, KG, kScratchBytes), M, K);
}

extern "C" int conv3d_fwd_split(const void* x, const void* w, const void* bias, const void* res,
                                void* out, int nB, int D, int H, int W, int C, int K, int T, int R,
                                int S, int sd, int sh, int sw, int Z, int P, int Q, long M,
                                long xsn, long xsd, long xsh, long xsw, long osn, long osz,
                                long osp, long osq, long rsn, long rsz, long rsp, long rsq,
                                hipStream_t stream, void* workspace, size_t workspace_bytes) {
    return conv3d_impl(x, w, bias, res, out, nB, D, H, W, C, K, T, R, S, sd, sh, sw, Z, P, Q, M,
                       xsn, xsd, xsh, xsw, osn, osz, osp, osq, rsn, rsz, rsp, rsq, stream,
                       workspace, workspace_bytes, false);
}

extern "C" void launch_conv3d(const void* x, const void* w, const void* bias, const void* res,
                              void* out, int nB, int D, int H, int W, int C, int K, int T, int R,
                              int S, int sd, int sh, int sw, int Z, int P, int Q, long M, long xsn,
                              long xsd, long xsh, long xsw, long osn, long osz, long osp, long osq,
                              long rsn, long rsz, long rsp, long rsq, hipStream_t stream) {
    (void)conv3d_fwd(x, w, bias, res, out, nB, D, H, W, C, K, T, R, S, sd, sh, sw, Z, P, Q, M, xsn,
                     xsd, xsh, xsw, osn, osz, osp, osq, rsn, rsz, rsp, rsq, stream);
}
