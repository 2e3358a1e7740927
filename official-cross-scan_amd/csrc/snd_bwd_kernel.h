// Backward kernel of the 2D-CrossScan selective scan for gfx950.
//
// Computes the gradients the reference's selective_scan_bwd_kernel produces
// (kernels/selective_nd_scan/include/cusoflex/selective_scan_bwd_kernel_oflex.cuh:91-902).
// With G = a*g, Gs = a*gs and every out-of-range term zero, per (batch, channel, state) plane:
//     g[i,j]  = dout*C + G[i,j+1] + G[i+1,j] - 0.5*(a[i,j+1] + a[i+1,j])*G[i+1,j+1]      (:463-469,486-488)
//     gs[i,j] = -dout*C + Gs[i,j+1]                                                      (:710,722-724)
//     dbu     = g + gs + 0.25*dout*C                                                     (:513,749-754)
//     da*a    = g*(h - bu) + gs*(s - bu) - 0.5*a*(G[i+1,j]*h[i,j-1] + G[i,j+1]*h[i-1,j]) (:515-587,751-753)
//     ddelta  = sum_n (A*da*a + dbu*B*u), then * sigmoid(raw) under softplus             (:516,752,785-806)
//     du      = D*dout + delta' * sum_n dbu*B                                            (:211,514,750)
//     dB      = sum_{c in group} dbu*delta'*u        dC = sum_{c in group} dout*(h - s + 0.25*bu)   (:589-590,754-755)
//     dA      = sum_{b,i,j} delta'*da*a              dD = sum dout*u     ddelta_bias = sum ddelta    (:518,753,212,808-819)
// (g*(h-bu) is the reference's dx*a with a = (h-bu); the two -0.5 terms are the places a[i,j]
// enters its right and lower neighbours, which the reference scatters to ddelta_vals[nrow-1][i],
// ddelta_vals[nrow][i-1] and stitches across chunk seams; here they are gathered at the cell.)
//
// Organisation (not a translation): the same lane = one (channel, state) plane, TE x TE tile walk
// as the forward (TE = 8 or 7), in reverse.  For each tile a lane recomputes h from the forward's checkpoints (row above
// from x_v, column to the left from x, s from x_sd) into 64 registers and sweeps the tile bottom-right to top-left.  The
// adjoint row handed to the strip above goes through a private global scratch row; the column handed to the tile on the
// left stays in registers.  dB/dC are reduced over a wave's channels with lane swaps, over the block's waves
// through LDS, and leave the block once per tile; du/ddelta are reduced over states by DPP and
// finished once per pixel by the thread that staged it.
// What the sweep evaluates per cell (22 vector instructions, and 7 for the sums over states and channels): the part of a lower
// row's contribution that does not depend on the row above it is formed where the row is swept, K = G - a/2 * G[right]; G + Gs is
// carried instead of Gs, since
//     g = dout*C + G[i,j+1] + K[i+1,j] - a[i,j+1]/2 * G[i+1,j+1]       g + gs = (G + Gs)[i,j+1] + K[i+1,j] - a[i,j+1]/2 * G[i+1,j+1]
// share their tail and dout*C cancels in the second; s - bu is a * s[left]; and the quarter terms of dB, dC and sum_n dbu*B are
// left to sums per pixel (flush_bc).  With the rest of a tile about 49 vector instructions per cell: two waves per SIMD issue
// them in 60 % of the kernel's time (64 x 192 x 56x56), the remainder are waits for operands, barriers and memory.
// As in the forward, tiles are computed in full on zero-padded staging (dout = B = C = 0 outside
// the plane makes every adjoint there exactly zero), so the inner loops have no bounds checks.
#pragma once
#include <initializer_list>
#include <type_traits>
#include "snd_device.h"

namespace snd {

// Pitch of the arrays that only the staging and the epilogue touch: with 16 states the 8x8 tiles leave LDS for no padding.
constexpr int bwd_pcs(int NP, int TE) { return kTile + (NP == 16 && TE == 8 ? 0 : NP < 8 ? NP : 8); }
// Exchange the upper 32 lanes of a with the lower 32 of b.
__device__ __forceinline__ void swap_halves(float &a, float &b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}

// Sum two sets of four values over the four 16-lane rows of a wave (its four channels when a row
// holds the 16 states of one channel): a reduce-scatter, row q of the wave ends with the totals of
// b[q] (in b0) and c[q] (in c0).  v_permlane32_swap exchanges the upper 32 lanes of its first
// operand with the lower 32 lanes of its second, v_permlane16_swap the odd 16-lane rows of the first
// with the even rows of the second; after either, first + second is the pair-sum of the value the
// lane keeps.  A swap must not read a register written by the two preceding VALU instructions and
// its results must not be read by the two following ones: the order and the s_nops keep that distance.
__device__ __forceinline__ void rows_scatter4x2(float &b0, float &b1, float &b2, float &b3, float &c0, float &c1,
                                                float &c2, float &c3) {
    asm volatile("s_nop 1\n\t"
                 "v_permlane32_swap_b32 %0, %2\n\t"
                 "v_permlane32_swap_b32 %1, %3\n\t"
                 "v_permlane32_swap_b32 %4, %6\n\t"
                 "v_permlane32_swap_b32 %5, %7\n\t"
                 "v_add_f32 %0, %0, %2\n\t"
                 "v_add_f32 %1, %1, %3\n\t"
                 "v_add_f32 %4, %4, %6\n\t"
                 "v_add_f32 %5, %5, %7\n\t"
                 "s_nop 0\n\t"
                 "v_permlane16_swap_b32 %0, %1\n\t"
                 "v_permlane16_swap_b32 %4, %5\n\t"
                 "s_nop 1\n\t"
                 "v_add_f32 %0, %0, %1\n\t"
                 "v_add_f32 %4, %4, %5\n\t"
                 : "+v"(b0), "+v"(b1), "+v"(b2), "+v"(b3), "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3));
}
// The two reductions of a half row in one block, for the 16-lane layout: group_scatter8 over q0..q3, p0..p3 (sums over the
// channel's 16 states) and rows_scatter4x2 over b0..b3, c0..c3 (sums over the wave's four channels).  The steps of one fill the
// slots that the other would spend on s_nops (a wave issues an s_nop as slowly as a multiply-add); both distances named above
// hold for every operand.
__device__ __forceinline__ void sweep_reduce16(float &q0, float &q1, float &q2, float &q3, float &p0, float &p1, float &p2, float &p3,
                                               float &b0, float &b1, float &b2, float &b3, float &c0, float &c1, float &c2, float &c3) {
    asm volatile("s_nop 1\n\t"
                 SND_DPPA("%0", "%0", "row_ror:8", "0x3") SND_DPPA("%1", "%1", "row_ror:8", "0x3")
                 SND_DPPA("%2", "%2", "row_ror:8", "0x3") SND_DPPA("%3", "%3", "row_ror:8", "0x3")
                 SND_DPPA("%0", "%4", "row_ror:8", "0xc") SND_DPPA("%1", "%5", "row_ror:8", "0xc")
                 SND_DPPA("%2", "%6", "row_ror:8", "0xc") SND_DPPA("%3", "%7", "row_ror:8", "0xc")
                 "v_permlane32_swap_b32 %8, %10\n\t"
                 "v_permlane32_swap_b32 %9, %11\n\t"
                 "v_permlane32_swap_b32 %12, %14\n\t"
                 "v_permlane32_swap_b32 %13, %15\n\t"
                 SND_DPPA("%0", "%0", "row_shl:4", "0x5") SND_DPPA("%1", "%1", "row_shl:4", "0x5")
                 SND_DPPA("%0", "%2", "row_shr:4", "0xa") SND_DPPA("%1", "%3", "row_shr:4", "0xa")
                 "v_add_f32 %8, %8, %10\n\t"
                 "v_add_f32 %9, %9, %11\n\t"
                 "v_add_f32 %12, %12, %14\n\t"
                 "v_add_f32 %13, %13, %15\n\t"
                 SND_DPPA("%0", "%0", "quad_perm:[1,0,3,2]", "0xf") SND_DPPA("%1", "%1", "quad_perm:[1,0,3,2]", "0xf")
                 "v_permlane16_swap_b32 %8, %9\n\t"
                 "v_permlane16_swap_b32 %12, %13\n\t"
                 SND_DPPA("%0", "%0", "quad_perm:[2,3,0,1]", "0xf") SND_DPPA("%1", "%1", "quad_perm:[2,3,0,1]", "0xf")
                 "v_add_f32 %8, %8, %9\n\t"
                 "v_add_f32 %12, %12, %13\n\t"
                 : "+v"(q0), "+v"(q1), "+v"(q2), "+v"(q3), "+v"(p0), "+v"(p1), "+v"(p2), "+v"(p3), "+v"(b0), "+v"(b1), "+v"(b2),
                   "+v"(b3), "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3));
}
// VEC: the tile's inputs are staged, and du / ddelta stored, four columns at a time with one 16-byte (fp32) or
// 8-byte (16-bit) access per thread and tensor instead of one access per element - a quarter of the memory
// instructions and of their address arithmetic.  Needs 8x8 tiles, a width that is a multiple of four and tensors
// whose rows start on such boundaries (bwd_vec_ok); everything else takes the element-wise staging.
// SEG: (pipelined strips only) a job is a column segment of a strip; the carried column state goes from one
// segment's block to the next through the workspace (strip_segments).  A variant of its own, because the few
// registers it takes are registers the other variants do not have.
// SINGLE: (whole planes) the plane is one tile: no tile follows whose inputs would be requested - the general kernel requests its own
// again - and nothing enters it, so no checkpoint is read.  64 x 1536 x 7x7 bf16, 16 states 174 -> 147 us, 64 x 768 x 7x7 fp16,
// 8 states 72 -> 60, 8 x 768 x 7x7 18.6 -> 16.1.  With four lanes per channel (up to 4 states) on 8x8 tiles it spills 29 registers
// where the general kernel spills none, and is the faster one all the same but for large fp32 launches: 64 x 3072 x 8x8, four states,
// bf16 208 -> 200, fp32 205 -> 207; 64 x 3072 x 7x8, two states, bf16 203 -> 192; 4 x 768 x 8x8, four, fp32 16.7 -> 15.9.  Branches around the requests instead: planes of several tiles lose up to 7 %
// (32 x 768 x 28x28 548 -> 586).
template <typename T, int NP, bool PIPE, int TE, bool VEC, bool SEG = false, bool SINGLE = false>
__global__ __launch_bounds__(16 * NP) __attribute__((amdgpu_waves_per_eu(2, 2))) void bwd_kernel(const snd_bwd_params p, const Geo geo) {
    static_assert(!VEC || TE == 8, "vector staging needs 8x8 tiles");
    static_assert(!SEG || PIPE, "column segments belong to the strip pipeline");
    static_assert(!SINGLE || !PIPE, "a plane of one tile has no strips");
    constexpr int WPB = NP / 4;                     // waves per block
    constexpr int CB = 16;                          // channels per block
    constexpr int NSTR = kTile + 4;
    // Pitches in floats, chosen for the 32 four-byte banks of LDS (a pitch of 64 would put every channel of a
    // wave in the same bank).  PCH: pixel arrays that the sweep reads as one float4 per channel (all lanes of a
    // channel the same address), so the channels of a wave must start 4 banks apart.  PCS: pixel arrays that
    // only the staging and the per-pixel epilogue touch, lane n of a channel at element n, so a channel takes NP
    // consecutive banks.  NSD: the dB/dC partial sums, which the 16-lane row q of a wave writes at element q of
    // a state's tile row, so states must start 2 (16 states) or 4 banks apart.
    constexpr int PCH = kTile + (NP == 16 ? 8 : 4);
    constexpr int PCS = bwd_pcs(NP, TE);
    constexpr int NSD = NP == 16 ? kTile + 2 : kTile + 4;
    constexpr int NBC = 4;
    constexpr int NPX = kTile / NP;
    // delta' on the tile plus a one-cell halo: rows -1..8 at a pitch of 12 floats, column j at element DLO + j, so
    // that columns 0-3 and 4-7 of a row are each one aligned 16-byte read (channels of a wave 24 banks apart)
    constexpr int HG = 12, DLO = 4, DLP = 10 * HG;
    constexpr int NHALO = 4 * TE + 4, NHK = (NHALO + NP - 1) / NP;   // ring around the TE x TE tile
    constexpr int NCH = VEC ? kTile / 4 / NP : 0;   // (VEC) four-column chunks of a channel's tile per thread
    constexpr int NHV = (24 + NP - 1) / NP;         // (VEC) halo cells per thread: row above, row below, column to the left

    // A wave's channels (four with 16 states per channel, eight with 8) are reduced in registers and
    // every wave owns a partial dB/dC tile, written with plain stores.
    constexpr int NPART = WPB;
    extern __shared__ __align__(16) float smem[];
    float *sB = smem;                               // [NP][NSTR]
    float *sC = sB + NP * NSTR;
    constexpr int PART = NP * NSD;
    float *sdB = sC + NP * NSTR;                    // [NPART][PART]
    float *sdC = sdB + NPART * PART;
    float *sDl = sdC + NPART * PART;                // [CB][DLP]
    float *sDu = sDl + CB * DLP;                    // [CB][PCH] delta' * u
    float *sQ = sDu;                                // sum_n dbu*B: takes the place of a row half's delta' * u once that is swept
    float *sU = sDu + CB * PCH;                     // [CB][PCS]
    float *sDo = sU + CB * PCS;                     // dout
    float *sSg = sDo + CB * PCH;                    // [CB][PCS] d softplus / d raw
    float *sP = sSg + CB * PCS + 4;                 // sum_n A*da*a (4 banks off sQ: a wave writes both in one instruction)
    float *sHold = sP + CB * PCH;                   // dB, dC sums of a pair's right tile, [2][NP][kTile]
    // sum over a wave's channels of dout * delta' * u / 4, [WPB][kTile], and sum over the states of B*C / 4, [kTile] (7x7 tiles
    // have no use for sHold)
    float *sT = TE == 7 ? sHold : sHold + 2 * NP * kTile, *sS = sT + WPB * kTile;
    float *sRed = sS + kTile;                       // [WPB]

    const snd_fwd_params &f = p.f;
    const snd_shape &sh = f.shape;
    const int H = sh.nrows, W = sh.ncols, N = sh.dstate, Dm = sh.dim, G = sh.n_groups;
    const int rg = Dm / G, rd = Dm / sh.delta_dim;
    const int nChunks = (rg + CB - 1) / CB;
    int pair, chunk;
    int I_hi = geo.nCY - 1, I_lo = 0;               // strips this block walks, bottom to top
    int J_hi = geo.nCX - 1, J_lo = 0, seg = 0;      // and the tiles of a strip, right to left (a column segment of a pipelined strip)
    int *sync = (int *)p.workspace, *progress = nullptr, *segdone = nullptr;
    float *colstate = nullptr;
    const int64_t nSync = sync_words((int64_t)sh.batch * G * nChunks, geo.nCY);
    bool dead = false;
    int seen = 0;                                   // last progress count read (strip pipeline)
    __shared__ int sSeen;                           // (pipelined) progress count of the strip below, as last polled
    __shared__ int sDead;                           // (pipelined) a hand-over wait of this block has timed out
    if (PIPE) {
        if (threadIdx.x == 0) { sSeen = 0; sDead = 0; }   // ordered before their readers by the barrier in draw_job
        // A job is a band of consecutive strips (one strip each in the fully pipelined case), drawn
        // bottom band first; band k from the bottom covers strips ceil(k*nCY/nBands) ..
        // ceil((k+1)*nCY/nBands)-1, counted from the bottom.
        int band;
        if (!draw_job(sync, sh.batch * G, nChunks, geo.nBands, geo.nQueues, pair, chunk, band, SEG ? geo.nSeg : 1, geo.segTiles, &seg)) return;
        const int nPC = sh.batch * G * nChunks;
        const int pc = pair * nChunks + chunk;
        I_hi = geo.nCY - 1 - (band * geo.nCY + geo.nBands - 1) / geo.nBands;
        I_lo = geo.nCY - ((band + 1) * geo.nCY + geo.nBands - 1) / geo.nBands;
        progress = sync + kSyncHeader + pc * geo.nCY;
        // (column-segmented strips: one strip per job) the segment's tiles, right to left; the carried column state
        // of the strip goes from segment to segment through one slot of the workspace
        if (SEG) {
            J_hi = geo.nCX - 1 - seg * geo.segTiles;
            J_lo = seg == geo.nSeg - 1 ? 0 : J_hi - geo.segTiles + 1;
            segdone = progress + nPC * geo.nCY;
            colstate = (float *)p.workspace + nSync + (int64_t)sh.batch * Dm * N * geo.Wp + ((int64_t)pc * geo.nCY + I_hi) * kColStateFloats;
        }
    } else if (!xcd_job(blockIdx.x, sh.batch * G, nChunks, pair, chunk)) return;
    const int b = pair / G, g = pair - b * G;
    const int cbase = g * rg + chunk * CB, cend = (g + 1) * rg;
    // scan origin of this group (as in the forward): memory row = mrow(i) = r0m + rs*i, column = mcol(j)
    const bool fv = f.directions == SND_DIR_CORNERS && (g & 2), fh = f.directions == SND_DIR_CORNERS && (g & 1);
    const int r0m = fv ? H - 1 : 0, rs = fv ? -1 : 1, c0m = fh ? W - 1 : 0, cs = fh ? -1 : 1;
    auto mrow = [&](int r) { return mad24(r, rs, r0m); };
    auto mcol = [&](int c_) { return mad24(c_, cs, c0m); };

    const int tid = threadIdx.x, wave = tid >> 6;
    const int n = tid % NP, cl = tid / NP;
    const int c = cbase + cl;
    const bool cvalid = c < cend;
    const bool lvalid = cvalid && n < N;
    const int cc = cvalid ? c : cend - 1, nn = n < N ? n : N - 1;
    const int px = tid & 63, pr = px >> 3, pj = px & 7;

    const float A2 = kLog2e * (lvalid ? f.A[(int64_t)cc * f.A_d_stride + (int64_t)nn * f.A_dstate_stride] : 0.f);
    const float ld = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, f.A_decay ? __log2f(f.A_decay[0]) : 0.f)));
    const float Dv = f.D ? f.D[cc] : 0.f;
    const float bias = f.delta_bias ? f.delta_bias[cc / rd] : 0.f;
    const bool softplus = f.delta_softplus != 0;

    // per-batch-image base pointers (uniform) and 32-bit offsets inside the image
    const T *Bb = (const T *)f.B + (int64_t)b * f.B_batch_stride + (int64_t)g * f.B_group_stride;
    const T *Cb = (const T *)f.C + (int64_t)b * f.C_batch_stride + (int64_t)g * f.C_group_stride;
    const T *ub = (const T *)f.u + (int64_t)b * f.u_batch_stride;
    const T *db = (const T *)f.delta + (int64_t)b * f.delta_batch_stride;
    const int sh_do = p.dout_dtype == SND_F32 ? 2 : 1, esz_do = 1 << sh_do;
    const void *dob = (const char *)p.dout + (int64_t)b * p.dout_batch_stride * esz_do;
    T *dub = (T *)p.du + (int64_t)b * Dm * H * W;                    // du, ddelta: dense [b, c, H, W]
    T *ddb = (T *)p.ddelta + (int64_t)b * Dm * H * W;
    float *dBg = p.dB + ((int64_t)b * G + g) * N * H * W;            // dense [b, g, N, H, W]
    float *dCg = p.dC + ((int64_t)b * G + g) * N * H * W;
    // byte offsets inside the batch image: per-lane channel offsets (kept across the tile loop) and
    // row pitches / state strides in bytes
    constexpr int ESZ = (int)sizeof(T);
    const uint32_t cUb = (uint32_t)(f.u_shared ? cc - g * rg : cc) * (uint32_t)f.u_d_stride * ESZ, cDb = (uint32_t)(cc / rd) * (uint32_t)f.delta_d_stride * ESZ;
    // fused CrossMerge: dout is the gradient of the merged output (one channel per feature, shared by the groups);
    // the channel's weight is applied where dout is staged, and every gradient, being linear in dout, follows
    const bool merge = f.merge != 0;
    // (times NaN if the saved state was written by the other kernel family: see kTagTile)
    const float wm = (merge && f.merge_weights ? f.merge_weights[cc] : 1.f) * tag_poison(geo.tag, kTagTile);
    const uint32_t cDob = ((uint32_t)(merge ? cc - g * rg : cc) * (uint32_t)p.dout_d_stride) << sh_do;
    const uint32_t cGb = (uint32_t)cc * (uint32_t)(H * W) * ESZ;      // du, ddelta
    const int BhB = (int)f.B_h_stride * ESZ, ChB = (int)f.C_h_stride * ESZ, UhB = (int)f.u_h_stride * ESZ, DhB = (int)f.delta_h_stride * ESZ;
    const int DohB = (int)p.dout_h_stride << sh_do, WB = W * ESZ, W4 = W * 4;
    const int64_t BsB = f.B_dstate_stride * ESZ, CsB = f.C_dstate_stride * ESZ;
    const int64_t HW4 = (int64_t)H * W * 4;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);   // the wave index as a scalar

    // saved state and scratch, tile-major; inside a tile the lanes' values 0-3, then the lanes' values
    // 4-7 (as the forward writes: a wave's 16-byte accesses cover whole lines):
    //   x_v [b][I][J][half][c][n][4 cols]   x, x_sd [b][J][I][half][c][n][4 rows]   scratch G row [b][J][half][c][n][4 cols]
    const int64_t DN8 = (int64_t)Dm * N * 8;
    const int64_t DN4 = DN8 / 2;
    // Addressed as a wave-uniform base (batch image, tile) plus one 32-bit byte offset per lane, laneB: one register for
    // all of them across the tile loop instead of a 64-bit pointer per array.
    const uint32_t laneB = (uint32_t)(cc * N + nn) * 16u;              // the lane's four floats inside a half tile
    const char *xv = (const char *)(f.x_v + (int64_t)b * geo.nCY * geo.nCX * DN8);
    const char *xh = (const char *)(f.x + (int64_t)b * geo.nCX * geo.nCY * DN8);
    const char *xs = (const char *)(f.x_sd + (int64_t)b * geo.nCX * geo.nCY * DN8);
    auto ck4 = [&](const char *tile, int64_t floats) __attribute__((always_inline)) {   // 16 bytes of this lane, `floats` into the tile
        return *(const float4 *)(tile + floats * 4 + laneB);
    };
    // hand-over between blocks (pipelined schedules): [J][pair k][c][n][2], so that a wave's 8-byte
    // coherent accesses cover whole lines too (the lane's offset there is half of laneB)
    const int64_t DN2 = (int64_t)Dm * N * 2;
    char *gdown = (char *)((float *)p.workspace + nSync + (int64_t)b * geo.nCX * DN8);
    const uint32_t laneG = PIPE ? laneB >> 1 : laneB;

    const float *myDl = sDl + cl * DLP;
    const float *myDu = sDu + cl * PCH;
    const float *myDo = sDo + cl * PCH;
    const float *myB = sB + n * NSTR;
    const float *myC = sC + n * NSTR;
    float *mydB = sdB + wave * NP * NSD + n * NSD;
    float *mydC = sdC + wave * NP * NSD + n * NSD;
    const int qrow = (tid & 63) >> 4;               // 16-lane row of this lane inside its wave
    float *myQP = ((n & 8) ? sP : sQ) + cl * PCH + ((n >> 1) & 2);   // (16 lanes) where this lane's quad leaves its sums over the states

    // ---- register staging of one tile's inputs: loaded in the second half of the sweep of the tile before, as they are, masked
    // and converted where they are committed to LDS
    uint32_t qb[VEC ? 1 : NBC], qc[VEC ? 1 : NBC], qdl[VEC ? 1 : NPX], qu[VEC ? 1 : NPX], qdo[VEC ? 1 : NPX], qh[VEC ? 1 : NHK];
    Raw4<T> vb, vc, vdl[VEC ? NCH : 1], vu[VEC ? NCH : 1];     // (VEC) one chunk of B and C, NCH chunks of delta, u, dout
    uint32_t vdo[VEC ? NCH : 1][4];
    uint32_t vh[VEC ? NHV : 1];
    // (VEC) halo cell k of this thread: cells 0-7 the row above, 8-15 the row below, 16-23 the column to the left
    auto halo_cell = [&](int hidx, int &rr, int &jj) {
        if (hidx < 8) { rr = -1; jj = hidx; }
        else if (hidx < 16) { rr = TE; jj = hidx - 8; }
        else { rr = hidx - 16; jj = -1; }
    };
    // (element-wise) cell k of the ring around the tile in the delta' grid, its coordinates relative to the tile
    auto ring_cell = [&](int hidx, int &rr, int &jj) {
        if (hidx < TE + 2) { rr = -1; jj = hidx - 1; }
        else if (hidx < 2 * TE + 4) { rr = TE; jj = hidx - (TE + 3); }
        else if (hidx < 3 * TE + 4) { rr = hidx - (2 * TE + 4); jj = -1; }
        else { rr = hidx - (3 * TE + 4); jj = TE; }
    };
    // Loads are always in bounds (clamped coordinates); commit() zeroes what lies outside the plane, the tile (7x7 tiles) and the
    // state / channel ranges.  part 0: B and C, 1: delta and u, 2: dout and the halo of delta.
    auto load_part = [&](int I, int J, int part) __attribute__((always_inline)) {
        const int r0 = I * TE, j0 = J * TE;
        // The thread's element maps are re-derived here from an opaque copy of the thread id, so that
        // they are a few integer ops per tile instead of dozens of registers kept live across the tile.
        SND_THREAD_MAPS(NP);
        if constexpr (VEC) {
            // Chunk q of a tile = row q / 2, columns 4 * (q % 2) .. + 3; under a mirrored column order the same four
            // memory columns in reverse (the chunk then starts at the memory column of its last scan column).
            auto chunk_off = [&](int q, int hB, int esz) {
                const int row = min(r0 + (q >> 1), H - 1), col = min(j0 + (q & 1) * 4, W - 4);
                return (uint32_t)mad24(mrow(row), hB, mcol(col + (fh ? 3 : 0)) * esz);
            };
            if (part == 0) {
                const int sn = min(t_ >> 4, N - 1), q = t_ & 15;
                ldraw4_b(vb, Bb, (uint32_t)sn * (uint32_t)BsB + chunk_off(q, BhB, ESZ));   // (below 2^32: bwd_vec_ok)
                ldraw4_b(vc, Cb, (uint32_t)sn * (uint32_t)CsB + chunk_off(q, ChB, ESZ));
            }
#pragma unroll
            for (int k = 0; k < NCH; ++k) {
                const int q = n + NP * k;
                if (part == 1) {
                    ldraw4_b(vdl[k], db, cDb + chunk_off(q, DhB, ESZ));
                    ldraw4_b(vu[k], ub, cUb + chunk_off(q, UhB, ESZ));
                } else if (part == 2) {
                    const char *src = (const char *)dob + (cDob + chunk_off(q, DohB, esz_do));
                    if (sizeof(T) == 4 || sh_do == 2) {
                        const uint4 v = *(const uint4 *)src;
                        vdo[k][0] = v.x; vdo[k][1] = v.y; vdo[k][2] = v.z; vdo[k][3] = v.w;
                    } else {
                        const uint2 v = *(const uint2 *)src;
                        vdo[k][0] = v.x; vdo[k][1] = v.y;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < (part == 2 ? NHV : 0); ++k) {
                int rr, jj;
                halo_cell(n + NP * k, rr, jj);
                const int row = min(max(r0 + rr, 0), H - 1), col = min(max(j0 + jj, 0), W - 1);
                vh[k] = ldraw_b(db, cDb + mad24(mrow(row), DhB, mcol(col) * ESZ));
            }
        } else {
            if (part == 0) {
                const int mr = mrow(min(r0 + pr, H - 1)), mcB = mcol(min(j0 + pj, W - 1)) * ESZ;
                const uint32_t ob = mad24(mr, BhB, mcB), oc = mad24(mr, ChB, mcB);
#pragma unroll
                for (int k = 0; k < NBC; ++k) {
                    const int sc = min(wave_u + WPB * k, N - 1);            // scalar: folded into the base
                    qb[k] = ldraw_b((const T *)((const char *)Bb + sc * BsB), ob);
                    qc[k] = ldraw_b((const T *)((const char *)Cb + sc * CsB), oc);
                }
            }
#pragma unroll
            for (int k = 0; k < NPX; ++k) {
                const int pp = n + NP * k;
                const int mr = mrow(min(r0 + (pp >> 3), H - 1)), mc = mcol(min(j0 + (pp & 7), W - 1));
                if (part == 1) {
                    qdl[k] = ldraw_b(db, cDb + mad24(mr, DhB, mc * ESZ));
                    qu[k] = ldraw_b(ub, cUb + mad24(mr, UhB, mc * ESZ));
                } else if (part == 2) {
                    const char *src = (const char *)dob + (cDob + mad24(mr, DohB, mc << sh_do));
                    qdo[k] = sizeof(T) == 4 || sh_do == 2 ? *(const uint32_t *)src : (uint32_t)*(const uint16_t *)src;
                }
            }
#pragma unroll
            for (int k = 0; k < (part == 2 ? NHK : 0); ++k) {
                int rr, jj;
                ring_cell(n + NP * k, rr, jj);
                qh[k] = ldraw_b(db, cDb + mad24(mrow(min(max(r0 + rr, 0), H - 1)), DhB, mcol(min(max(j0 + jj, 0), W - 1)) * ESZ));
            }
        }
    };
    auto commit = [&](int I, int J) {
        SND_THREAD_MAPS(NP);
        if constexpr (VEC) {
            const int r0 = I * TE, j0 = J * TE;
            auto flip4 = [&](float (&v)[4]) {                     // memory order -> scan order under a mirrored column order
                if (fh) { const float a0 = v[0], a1 = v[1]; v[0] = v[3]; v[1] = v[2]; v[2] = a1; v[3] = a0; }
            };
            {
                const int sn = t_ >> 4, q = t_ & 15;
                const bool ok = sn < N && r0 + (q >> 1) < H && j0 + (q & 1) * 4 < W;
                float b4[4], c4[4];
                raw4_to_f32(vb, b4); raw4_to_f32(vc, c4);
                flip4(b4); flip4(c4);
#pragma unroll
                for (int e = 0; e < 4; ++e) { b4[e] = ok ? b4[e] : 0.f; c4[e] = ok ? c4[e] : 0.f; }
                *(float4 *)(sB + sn * NSTR + q * 4) = make_float4(b4[0], b4[1], b4[2], b4[3]);
                *(float4 *)(sC + sn * NSTR + q * 4) = make_float4(c4[0], c4[1], c4[2], c4[3]);
            }
#pragma unroll
            for (int k = 0; k < NCH; ++k) {
                const int q = n + NP * k;
                const bool ok = cvalid && r0 + (q >> 1) < H && j0 + (q & 1) * 4 < W;
                float d4[4], u4[4], o4[4], dl4[4], du4[4], sg4[4];
                raw4_to_f32(vdl[k], d4); raw4_to_f32(vu[k], u4);
                if (sizeof(T) == 4 || sh_do == 2) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) o4[e] = __builtin_bit_cast(float, vdo[k][e]);
                } else {
                    Raw4<T> t4;
                    t4.w[0] = vdo[k][0]; t4.w[sizeof(T) == 4 ? 0 : 1] = vdo[k][1];
                    raw4_to_f32(t4, o4);
                }
                flip4(d4); flip4(u4); flip4(o4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float raw = (ok ? d4[e] : 0.f) + bias;
                    float dsp = 1.f;
                    dl4[e] = softplus ? softplus20(raw, dsp) : raw;
                    u4[e] = ok ? u4[e] : 0.f;
                    du4[e] = dl4[e] * u4[e];
                    o4[e] = ok ? wm * o4[e] : 0.f;
                    sg4[e] = dsp;
                }
                *(float4 *)(sDl + cl * DLP + ((q >> 1) + 1) * HG + DLO + (q & 1) * 4) = make_float4(dl4[0], dl4[1], dl4[2], dl4[3]);
                *(float4 *)(sDu + cl * PCH + q * 4) = make_float4(du4[0], du4[1], du4[2], du4[3]);
                *(float4 *)(sU + cl * PCS + q * 4) = make_float4(u4[0], u4[1], u4[2], u4[3]);
                *(float4 *)(sDo + cl * PCH + q * 4) = make_float4(o4[0], o4[1], o4[2], o4[3]);
                *(float4 *)(sSg + cl * PCS + q * 4) = make_float4(sg4[0], sg4[1], sg4[2], sg4[3]);
            }
#pragma unroll
            for (int k = 0; k < NHV; ++k) {
                const int hidx = n + NP * k;
                int rr, jj;
                halo_cell(hidx, rr, jj);
                const bool ok = cvalid && r0 + rr >= 0 && r0 + rr < H && j0 + jj >= 0 && j0 + jj < W;
                const float raw = (ok ? raw_to_f32((const T *)nullptr, vh[k]) : 0.f) + bias;
                float dsp;
                if (hidx < 24) sDl[cl * DLP + (rr + 1) * HG + DLO + jj] = softplus ? softplus20(raw, dsp) : raw;
            }
            return;
        }
        const int r0 = I * TE, j0 = J * TE;
        {
            const bool in = pr < TE && pj < TE && r0 + pr < H && j0 + pj < W;
#pragma unroll
            for (int k = 0; k < NBC; ++k) {
                const int sn = wave + WPB * k;
                const bool ok = in && wave_u + WPB * k < N;
                sB[sn * NSTR + px] = ok ? raw_to_f32((const T *)nullptr, qb[k]) : 0.f;
                sC[sn * NSTR + px] = ok ? raw_to_f32((const T *)nullptr, qc[k]) : 0.f;
            }
        }
#pragma unroll
        for (int k = 0; k < NPX; ++k) {
            const int pp = n + NP * k;
            const bool ok = cvalid && (pp >> 3) < TE && (pp & 7) < TE && r0 + (pp >> 3) < H && j0 + (pp & 7) < W;
            const float raw = (ok ? raw_to_f32((const T *)nullptr, qdl[k]) : 0.f) + bias, u_ = ok ? raw_to_f32((const T *)nullptr, qu[k]) : 0.f;
            const float do_ = sizeof(T) == 4 || sh_do == 2 ? __builtin_bit_cast(float, qdo[k]) : raw_to_f32((const T *)nullptr, qdo[k]);
            float dsp = 1.f;
            const float dl = softplus ? softplus20(raw, dsp) : raw;
            if (TE == 8 || ((pp >> 3) < TE && (pp & 7) < TE))     // slots beyond the tile belong to the halo ring
                sDl[cl * DLP + ((pp >> 3) + 1) * HG + DLO + (pp & 7)] = dl;
            sDu[cl * PCH + pp] = dl * u_;
            sU[cl * PCS + pp] = u_;
            sDo[cl * PCH + pp] = ok ? wm * do_ : 0.f;
            sSg[cl * PCS + pp] = dsp;
        }
#pragma unroll
        for (int k = 0; k < NHK; ++k) {
            const int hidx = n + NP * k;
            int rr, jj;
            ring_cell(hidx, rr, jj);
            const bool ok = cvalid && hidx < NHALO && r0 + rr >= 0 && r0 + rr < H && j0 + jj >= 0 && j0 + jj < W;
            const float raw = (ok ? raw_to_f32((const T *)nullptr, qh[k]) : 0.f) + bias;
            float dsp;
            if (hidx < NHALO && DLO + jj < HG)          // (the column right of an 8-column tile is never read)
                sDl[cl * DLP + (rr + 1) * HG + DLO + jj] = softplus ? softplus20(raw, dsp) : raw;
        }
    };
#define DL(r, j) myDl[((r) + 1) * HG + DLO + (j)]
#define AEXP(r, j) EXPA(DL(r, j))
    // delta' of columns c0 .. c0+3 (c0 = 0 or 4) of tile row r (-1 .. 8): one aligned 16-byte read
    auto dl_row4 = [&](int r, int c0, float (&o)[4]) __attribute__((always_inline)) {
        const float4 v = *(const float4 *)(myDl + (r + 1) * HG + DLO + c0);
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    };
#define EXPA(x) fast_exp2(fmaf((x), A2, ld))

    float dA_acc = 0.f, dec_acc = 0.f;              // per lane: sum delta'*da*a, sum da*a
    const bool want_decay = p.dA_decay != nullptr;  // the second sum is skipped when nobody reads it
    float dD_acc = 0.f, dbias_acc = 0.f;            // per thread, for its channel's staged pixels
    // Fused CrossMerge: weight * d(weight) = <weighted dout, result of the channel>.  The result is linear in u
    // (D*u plus a recurrence that is linear in B*delta'*u), so this inner product equals <du, u>: summed per pixel
    // beside dD, at no cost in the sweep.
    float dw_acc = 0.f;

    // dB, dC of a tile leave the block (summed over its channels) behind its sweep and epilogue, from the waves' partial sums in LDS:
    // a tenth of a tile's time.  One tile late, ahead of the next tile's commit, with the zeros of border tiles ahead of it too and
    // loads in flight on the way into the tile loop (below), us: 64 x 192 x 56x56 fp32 1080 -> 1049, 2 x 192 x 200x336 922 -> 884, 1 x 256 x
    // 512^2 bf16 1993 -> 1968, 8 x 768 x 56x56 bf16 556 -> 539, 12 x 196 x 65x91 657 -> 630, 64 x 1536 x 7x7 144 -> 135.  They are read
    // (flush_read) ahead of the epilogue, under which the reads arrive: 0 to 0.5 % faster than behind it.  (The atomics one state at a time
    // between the rows of the next recomputation: 1.3 to 4 % slower than all at once, with those of held tiles dropped by their offset.
    // A column segment's hand-over ahead of the last tile's flush instead of behind it: 2 x 192 x 200x336 fp32 878 -> 885, 4 x 96 x 256x256
    // 940 -> 939, 2 x 384 x 100x168 fp16 463 -> 493.)
    // The terms in dout*C/4 and bu/4 are left out of the sweep: summed over channels (states) they are products of B or C
    // with per-pixel sums that all states (channels) share,
    //     dB: C * T,  dC: B * T,  T = sum_c dout*delta'*u / 4        sum_n dbu*B: dout * S,  S = sum_n B*C / 4
    // That and s - bu = a * s[left] take four instructions per cell out of the sweep.
    // (All schedules alike, so that their results agree bit for bit.)
    float pB[NBC], pC[NBC];                         // this thread's B, C of the tile
    // Two neighbouring 8x8 tiles leave together: the right one's sums are held in LDS and joined to the left one's, so that an
    // instruction adds 4 rows x 16 columns instead of 8 rows x 8.  An atomic costs its CU 12 ns per 64-byte line it
    // touches, however few of the line's words it adds to (2 x 192 x 200x336: 1.09 -> 1.07 ms, 256 channels of 512x512:
    // 2.56 -> 2.51 ms; rows that are no multiple of 64 bytes gain nothing, 7x7 tiles lose 2 % and keep the plain form).
    // Lanes outside the plane get an offset that the buffer's range check drops: no branch around an atomic.
    struct Part { float t[WPB], b[NBC][NPART], c[NBC][NPART]; };
    auto flush_read = [&](Part &q) __attribute__((always_inline)) {
        SND_THREAD_MAPS(NP);
#pragma unroll
        for (int w = 0; w < WPB; ++w) q.t[w] = sT[w * kTile + px];
#pragma unroll
        for (int k = 0; k < NBC; ++k)
#pragma unroll
            for (int w = 0; w < NPART; ++w) {
                q.b[k][w] = sdB[w * PART + (wave_u + WPB * k) * NSD + px];
                q.c[k][w] = sdC[w * PART + (wave_u + WPB * k) * NSD + px];
            }
    };
    auto flush_bc = [&](const Part &q, int I, int J) __attribute__((always_inline)) {
        SND_THREAD_MAPS(NP);
        const bool holds = TE == 8 && (J & 1) && J > J_lo, joins = TE == 8 && !(J & 1) && J < J_hi;
        // plain: lane l adds row l / 8, column l % 8; joined: row (l / 8) % 4 (+ 4), column l % 8 of the left (lanes 0-31) or right tile
        const int row = I * TE + (joins ? pr & 3 : pr), col = (J + (joins ? px >> 5 : 0)) * TE + pj;
        const bool in = pr < TE && pj < TE && col < W;
        const int cB = mcol(col) * 4;
        const uint32_t o0 = in && row < H ? (uint32_t)mad24(mrow(row), W4, cB) : kBufOOB;
        const uint32_t o4 = in && row + 4 < H ? (uint32_t)mad24(mrow(row + 4), W4, cB) : kBufOOB;
        float tsum = 0.f;
#pragma unroll
        for (int w = 0; w < WPB; ++w) tsum += q.t[w];
#pragma unroll
        for (int k = 0; k < NBC; ++k) {
            int sn = wave_u + WPB * k;              // scalar: folded into the base
            asm volatile("" : "+s"(sn));            // (not eight descriptors kept across the tile loop)
            float tb = pC[k] * tsum, tc = pB[k] * tsum;
#pragma unroll
            for (int w = 0; w < NPART; ++w) {
                tb += q.b[k][w];
                tc += q.c[k][w];
            }
            if (holds) {
                sHold[sn * kTile + px] = tb;
                sHold[(NP + sn) * kTile + px] = tc;
            } else if (sn < N) {
                const __amdgpu_buffer_rsrc_t rB = buf_rsrc((char *)dBg + sn * HW4), rC = buf_rsrc((char *)dCg + sn * HW4);
                if (joins) {
                    // left tile: tb, right tile: what is held.  The swap exchanges the upper half of the first (rows 4-7 of the
                    // left tile) with the lower half of the second (rows 0-3 of the right one): rows 0-3 of both, rows 4-7 of both.
                    float hb = sHold[sn * kTile + px], hc_ = sHold[(NP + sn) * kTile + px];
                    swap_halves(tb, hb);
                    swap_halves(tc, hc_);
                    buf_add_f32(rB, o0, 0, tb);
                    buf_add_f32(rB, o4, 0, hb);
                    buf_add_f32(rC, o0, 0, tc);
                    buf_add_f32(rC, o4, 0, hc_);
                } else {
                    buf_add_f32(rB, o0, 0, tb);
                    buf_add_f32(rC, o0, 0, tc);
                }
            }
        }
    };
    // ---- checkpoints of a tile (h of the row above, h and s of the column to the left), loaded like its inputs in the sweep of the
    // tile before it; clamped to the plane, zeroed where they are needed
    float hu[kCkX], hlft[kRows], slft[kRows], hc = 0.f;
    auto load_row_ckpt = [&](int I, int J) __attribute__((always_inline)) {
        const char *src = xv + ((int64_t)max(I - 1, 0) * geo.nCX + J) * DN8 * 4;
        const float4 v0 = ck4(src, 0), v1 = ck4(src, DN4);
        hu[0] = v0.x; hu[1] = v0.y; hu[2] = v0.z; hu[3] = v0.w;
        hu[4] = v1.x; hu[5] = v1.y; hu[6] = v1.z; hu[7] = v1.w;
        // last column of the tile on the left
        hc = *(const float *)(src + (J > 0 ? (((TE - 1) >> 2) * DN4 + ((TE - 1) & 3) - DN8) * 4 : 0) + laneB);
    };
    auto load_col_ckpt = [&](int I, int J) __attribute__((always_inline)) {
        const int64_t t_ = ((int64_t)max(J - 1, 0) * geo.nCY + I) * DN8 * 4;
        const float4 h0 = ck4(xh + t_, 0), h1 = ck4(xh + t_, DN4);
        const float4 s0 = ck4(xs + t_, 0), s1 = ck4(xs + t_, DN4);
        hlft[0] = h0.x; hlft[1] = h0.y; hlft[2] = h0.z; hlft[3] = h0.w;
        hlft[4] = h1.x; hlft[5] = h1.y; hlft[6] = h1.z; hlft[7] = h1.w;
        slft[0] = s0.x; slft[1] = s0.y; slft[2] = s0.z; slft[3] = s0.w;
        slft[4] = s1.x; slft[5] = s1.y; slft[6] = s1.z; slft[7] = s1.w;
    };
    load_part(I_hi, J_hi, 0);
    load_part(I_hi, J_hi, 1);
    load_part(I_hi, J_hi, 2);
    if (!SINGLE) {
        load_row_ckpt(I_hi, J_hi);
        load_col_ckpt(I_hi, J_hi);
    }
    // Nothing in flight on the way into the tile loop: the waits that the compiler derives for the staged inputs then count the loop's own
    // instructions behind them instead of waiting for all of them.  Whole planes of several tiles lose by it (64 x 768 x 14x14 277 ->
    // 279 us, 32 x 768 x 28x28 541 -> 551).
    if (PIPE || SINGLE) __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    for (int I = I_hi; I >= I_lo; --I) {
        const int r0 = I * TE;
        float GR[kRows], SR[kRows];                 // G, G + Gs at the column right of the tile
        float tR[kRows];                            // -a/2 at that column (only ever multiplies G there)
        float GRc = 0.f;                            // G[r0+8][j0+8]
#pragma unroll
        for (int r = 0; r < kRows; ++r) { GR[r] = 0.f; SR[r] = 0.f; tR[r] = 0.f; }
        if (SEG && seg > 0) {
            // a later column segment of the strip: G, G + Gs, -a/2 of the column right of it and the corner G come from the
            // block that swept the segment before (written in full before its count moved: see strip_stores_done)
            if (wave == 0) {
                int seen_ = 0;
                strip_wait(segdone + I, seg, seen_, sync, dead, geo.spinLimit);
                if (dead && tid == 0) sDead = 1;
            }
            __syncthreads();
            const float *src = colstate + (tid << 1);
            const bool bad = lds_peek(&sDead) != 0;   // the wait timed out: poison everything downstream
#pragma unroll
            for (int r = 0; r < kRows; r += 2) {
                ld2_coherent(src + (r >> 1) * 512, GR[r], GR[r + 1]);
                ld2_coherent(src + (4 + (r >> 1)) * 512, SR[r], SR[r + 1]);
                ld2_coherent(src + (8 + (r >> 1)) * 512, tR[r], tR[r + 1]);
            }
            float pad_;
            ld2_coherent(src + 12 * 512, GRc, pad_);
            if (bad) {
                GRc = __builtin_nanf("");
#pragma unroll
                for (int r = 0; r < kRows; ++r) GR[r] = SR[r] = __builtin_nanf("");
            }
        }

        for (int J = SEG ? J_hi : geo.nCX - 1; J >= (SEG ? J_lo : 0); --J) {
            const int j0 = J * TE;
            // the next tile (the block's last: loads that nobody reads, of a tile that exists)
            int In = I, Jn = J - 1;
            if (Jn < (SEG ? J_lo : 0)) { In = I - 1; Jn = J_hi; }
            if (In < I_lo) { In = I; Jn = J; }
            float Gd[kCkX];                                        // G of the row below
            // the adjoint row of the strip below: written by this block, or - first strip of a
            // pipelined band - by another block.  It is requested here if it is known to be there (own
            // rows; rows whose hand-over an earlier poll has already seen), else after the wait below.
            const bool handed = PIPE && I == I_hi && I + 1 < geo.nCY;
            auto take_row = [&](int J_) __attribute__((always_inline)) {   // (pipelined schedules: through coherent words)
                if (!SINGLE && I + 1 < geo.nCY && lvalid) {
                    const char *src = gdown + (int64_t)J_ * DN8 * 4;
                    if (PIPE) {
#pragma unroll
                        for (int k = 0; k < kCkX; k += 2) ld2_coherent((const float *)(src + (k >> 1) * DN2 * 4 + laneG), Gd[k], Gd[k + 1]);
                    } else {
                        const float4 v0 = *(const float4 *)(src + laneG), v1 = *(const float4 *)(src + DN4 * 4 + laneG);
                        Gd[0] = v0.x; Gd[1] = v0.y; Gd[2] = v0.z; Gd[3] = v0.w;
                        Gd[4] = v1.x; Gd[5] = v1.y; Gd[6] = v1.z; Gd[7] = v1.w;
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < kCkX; ++j) Gd[j] = 0.f;
                }
            };
            const bool late = handed && __builtin_amdgcn_readfirstlane(lds_peek(&sSeen)) < geo.nCX - J;
            int peek = 0;                           // wave 0: the count as it is now, there when the staged inputs are
            if (late && wave == 0) peek = __hip_atomic_load(progress + I + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            commit(I, J);
            if (late && wave == 0) {
                seen = __builtin_amdgcn_readfirstlane(peek);
                if (tid == 0) lds_poke(&sSeen, dead ? geo.nCX : seen);
            }
            __syncthreads();
            const bool soon = late && __builtin_amdgcn_readfirstlane(lds_peek(&sSeen)) >= geo.nCX - J;
            {
                // T of this wave's channels (only this wave touches their delta' * u, whose place the sweep reuses), and S:
                // the pixels dealt over the waves, the states over the lanes of a pixel
                const int lane = tid & 63;
                float t = 0.f, v = 0.f;
#pragma unroll
                for (int k = 0; k < CB / WPB; ++k) t = fmaf(sDu[(wave_u * (CB / WPB) + k) * PCH + lane], sDo[(wave_u * (CB / WPB) + k) * PCH + lane], t);
                sT[wave_u * kTile + lane] = 0.25f * t;
                constexpr int PXW = kTile / WPB;
                const int spx = PXW * wave_u + lane % PXW;
#pragma unroll
                for (int k = 0; k < 4; ++k) v = fmaf(sB[(lane / PXW * 4 + k) * NSTR + spx], sC[(lane / PXW * 4 + k) * NSTR + spx], v);
#pragma unroll
                for (int m = PXW; m < 64; m <<= 1) v += __shfl_xor(v, m);
                if (lane < PXW) sS[spx] = 0.25f * v;
            }
            // (nothing enters the first row and column of tiles; here and not sooner, since it waits for the checkpoints requested)
            if (SINGLE || I == 0) {
#pragma unroll
                for (int j = 0; j < kCkX; ++j) hu[j] = 0.f;
                hc = 0.f;
            }
            if (SINGLE || J == 0) {
#pragma unroll
                for (int r = 0; r < kRows; ++r) { hlft[r] = 0.f; slft[r] = 0.f; }
                hc = 0.f;
            }
            // ---- recompute h on the whole tile, and s at column 3 of every row (the sweep takes a row's right half first)
            float hT[TE][TE], smid[TE];
            // columns whose a is kept from this pass for the sweep: as many as fit under 256 registers without a spill in
            // the tile loop (a spilled register is two vector memory instructions per tile, 2 to 4 % of the kernel); the column
            // segments' bookkeeping leaves room for two, a 7x7 tile for all (four / seven, bf16, us: 64 x 768 x 14x14 280 / 277, 32 x 768 x 28x28
            // 551 / 541, 64 x 1536 x 7x7 137 / 135; in its pipelined form four, with no difference between the two that builds alike do not show,
            // 16 x 384 x 21x35 fp32 175 to 185).
            constexpr int KA = TE == 7 ? (PIPE ? 4 : 7) : SEG ? 2 : 5;
            float aT[KA ? TE : 1][KA ? KA : 1];
            {
                float aprev[8], hprev[8], dlr[4];
#pragma unroll
                for (int c0 = 0; c0 < 8; c0 += 4) {
                    dl_row4(-1, c0, dlr);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (c0 + j < TE) { aprev[c0 + j] = EXPA(dlr[j]); hprev[c0 + j] = hu[c0 + j]; }
                }
                float diag0 = hc;
                // (a half row's operands are requested ahead of the arithmetic of the half row before it)
                float4 nD = *(const float4 *)(myDl + HG + DLO), nB = *(const float4 *)myB, nU = *(const float4 *)myDu;
                float nl = DL(0, -1);
#pragma unroll
                for (int r = 0; r < TE; ++r) {
                    if (r == 2 && (!late || soon)) take_row(J);    // it arrives under the rest of the recomputation
                    float al = EXPA(nl), left = hlft[r], sl = slft[r], diag = diag0;
                    diag0 = hlft[r];
#pragma unroll
                    for (int c0 = 0; c0 < 8; c0 += 4) {
                        const float aD[4] = {nD.x, nD.y, nD.z, nD.w}, aB[4] = {nB.x, nB.y, nB.z, nB.w}, aU[4] = {nU.x, nU.y, nU.z, nU.w};
                        __builtin_amdgcn_sched_barrier(0);
                        if (c0 == 0 || r + 1 < TE) {
                            const int nr = c0 == 0 ? r : r + 1, nc = 4 - c0;
                            nD = *(const float4 *)(myDl + (nr + 1) * HG + DLO + nc);
                            nB = *(const float4 *)(myB + nr * kCkX + nc);
                            nU = *(const float4 *)(myDu + nr * kCkX + nc);
                            if (c0) nl = DL(nr, -1);
                        }
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int c_ = c0 + j;
                            if (c_ >= TE) continue;
                            const float a = EXPA(aD[j]);
                            const float bu = aB[j] * aU[j];
                            const float up = hprev[c_];
                            const float X = fmaf(-0.5f * (aprev[c_] + al), diag, up);
                            const float h = fmaf(a, left + X, bu);
                            if (c0 == 0) sl = fmaf(a, sl, bu);
                            hT[r][c_] = h;
                            if (c_ < KA) aT[KA ? r : 0][KA ? c_ : 0] = a;
                            hprev[c_] = h;
                            diag = up; left = h; al = a; aprev[c_] = a;
                        }
                    }
                    smid[r] = sl;
                    // (computed here: left alone the compiler moves arithmetic that only the sweep reads behind the branches between,
                    // and holds its operands, twice the registers, until then)
                    asm volatile("" : "+v"(smid[r]));
#pragma unroll
                    for (int j = 0; j < TE; ++j) {
                        asm volatile("" : "+v"(hT[r][j]));
                        hprev[j] = hT[r][j];
                        if (j < KA) {
                            asm volatile("" : "+v"(aT[r][j]));
                            aprev[j] = aT[r][j];
                        }
                    }
                }
            }
            // strip pipeline: the strip below must have handed over tile J - wanted here, behind the recomputation, and no sooner.
            // One wave polls the count in memory (more pollers only slow it down), the others the word it leaves in LDS.
            // Waiting ahead of the recomputation cost 1.5-7 % of the pipelined backwards: 1 x 256 x 512^2 bf16, 16 states
            // 2396 -> 2328 us; 2 x 192 x 200x336 fp32 1063 -> 1040; 3 x 152 x 61x83 fp16, 8 states 225 -> 209 (unpipelined: same).
            if (late && !soon && wave == 0) {
                strip_wait(progress + I + 1, geo.nCX - J, seen, sync, dead, geo.spinLimit);
                if (tid == 0) {
                    if (dead) sDead = 1;
                    lds_poke(&sSeen, dead ? geo.nCX : seen);   // (read at the top of later tiles, too)
                }
            }
            if (PIPE) __syncthreads();              // the row below is there
            if (late && !soon) take_row(J);
            if (handed && lds_peek(&sDead)) {   // the wait timed out: poison everything downstream
#pragma unroll
                for (int j = 0; j < kCkX; ++j) Gd[j] = __builtin_nanf("");
            }
            const float gd_old0 = Gd[0];            // G[r0+8][j0]: the corner of the tile on the left
            // ---- reverse sweep, bottom-right to top-left.  K[j] = G[j] - 0.5*a[j]*G[j+1] of the row below: the part of its
            // contribution to g that does not depend on this row.
            float Kd[8];
            asm volatile("" ::: "memory");
            {
                float dlr[4];
#pragma unroll
                for (int c0 = 0; c0 < 8; c0 += 4) {
                    dl_row4(TE, c0, dlr);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (c0 + j < TE) Kd[c0 + j] = fmaf(-0.5f * EXPA(dlr[j]), c0 + j + 1 < TE ? Gd[c0 + j + 1 < 8 ? c0 + j + 1 : 7] : GRc, Gd[c0 + j]);
                }
            }
            // The sweep runs at a raised wave priority, everything else (loads, commit to LDS, recomputation, per-pixel epilogue)
            // at the default: the two waves a SIMD holds belong to two blocks, and with equal priority they drift into the same
            // phase and stall together; with the wave that is in its long arithmetic preferred, the other's phases fall into its
            // gaps.  Backward in us, raised from the recomputation on / raised for the sweep alone: 64 x 192 x
            // 56x56 fp32 1064 / 1057, 1 x 256 x 512^2 bf16 2072 / 1998, 32 x 768 x 28x28 bf16 575 / 551, 64 x 768 x
            // 14x14 291 / 286, 2 x 192 x 200x336 916 / 915.  Middle levels for the recomputation or the memory phases: alike.
            __builtin_amdgcn_s_setprio(3);
            float Gd8 = GRc;                        // G[r+1][j0+TE]
            // a half row's operands are requested ahead of the reductions of the half row before it, under which they arrive
            float4 nD4, nB4, nU4, nC4, nO4;
            auto half_row = [&](int r, int C0) __attribute__((always_inline)) {
                nD4 = *(const float4 *)(myDl + (r + 1) * HG + DLO + C0); nB4 = *(const float4 *)(myB + r * kCkX + C0);
                nU4 = *(const float4 *)(myDu + r * kCkX + C0); nC4 = *(const float4 *)(myC + r * kCkX + C0);
                nO4 = *(const float4 *)(myDo + r * kCkX + C0);
            };
            half_row(TE - 1, 4);
#pragma unroll
            for (int r = TE - 1; r >= 0; --r) {
                // the next tile's loads, between the rows of the second half, where the registers of the rows swept are free
                if (!SINGLE && r == 4) load_part(In, Jn, 0);
                if (!SINGLE && r == 3) load_part(In, Jn, 1);
                if (!SINGLE && r == 2) load_part(In, Jn, 2);
                float Gr = GR[r], Sr = SR[r], Gdiag = Gd8, tr = tR[r];
#pragma unroll
                for (int C0 = 4; C0 >= 0; C0 -= 4) {
                    __builtin_amdgcn_sched_barrier(0);
                    const int HW = C0 == 0 ? 4 : TE - 4;        // columns of this half inside the tile
                    const float dlr[4] = {nD4.x, nD4.y, nD4.z, nD4.w}, aB[4] = {nB4.x, nB4.y, nB4.z, nB4.w}, aC[4] = {nC4.x, nC4.y, nC4.z, nC4.w};
                    const float aU[4] = {nU4.x, nU4.y, nU4.z, nU4.w}, aO[4] = {nO4.x, nO4.y, nO4.z, nO4.w};
                    float arow[4], s[4], sbv[4] = {};
                    float sp = C0 ? smid[r] : slft[r];
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (j < HW) {
                            arow[j] = C0 + j < KA ? aT[KA ? r : 0][C0 + j < KA ? C0 + j : 0] : EXPA(dlr[j]);
                            sbv[j] = arow[j] * sp;                 // s - bu
                            sp = fmaf(aB[j], aU[j], sbv[j]);
                            s[j] = sp;
                        }
                    float q[4] = {}, pp_[4] = {}, vB[4] = {}, vC[4] = {}, dsum[4] = {};
#pragma unroll
                    for (int j = 3; j >= 0; --j) {
                        if (j >= HW) continue;
                        const int cj = C0 + j;
                        const float dov = aO[j], duv = aU[j], a = arow[j];
                        const float w = fmaf(tr, Gdiag, Kd[cj]);
                        const float g_ = fmaf(dov, aC[j], w + Gr), gg = w + Sr;   // g, and g + gs (dout*C cancels)
                        const float h_l = cj == 0 ? hlft[r] : hT[r][cj - 1 < 0 ? 0 : cj - 1];
                        const float h_u = r == 0 ? hu[cj] : hT[r - 1 < 0 ? 0 : r - 1][cj];
                        // g(h - bu) + gs(s - bu) = g(h - s) + (g + gs)(s - bu)
                        const float hs = hT[r][cj] - s[j];
                        const float cross = fmaf(Gd[cj], h_l, Gr * h_u);
                        const float t = -0.5f * a;
                        const float da = fmaf(t, cross, fmaf(g_, hs, gg * sbv[j]));
                        dA_acc = fmaf(dlr[j], da, dA_acc);
                        dsum[j] = da;
                        const float Gn = a * g_;
                        Gdiag = Gd[cj];
                        Kd[cj] = fmaf(t, Gr, Gn);
                        Gd[cj] = Gn;
                        Gr = Gn;
                        Sr = a * gg;
                        tr = t;
                        q[j] = gg * aB[j];                         // per-pixel terms, summed over states below
                        pp_[j] = A2 * da;
                        vB[j] = gg * duv;                          // dB, dC contributions
                        vC[j] = dov * hs;
                    }
                    if (want_decay) {
                        dec_acc += (dsum[0] + dsum[1]) + (dsum[2] + dsum[3]);
                        asm volatile("" : "+v"(dec_acc));
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (C0) half_row(r, 0);
                    else if (r > 0) half_row(r - 1, 4);
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("" : "+v"(dA_acc));    // (added up here: left alone the compiler keeps the terms of the whole tile for its end)
                    if (NP == 16) {
                        // sums over the channel's 16 states: quads 0,1 of the lane group end with
                        // q[0..1], q[2..3], quads 2,3 with pp_[0..1], pp_[2..3] (a quad's four lanes write the same words);
                        // over the wave's channels: the 16-lane row q ends with column C0+q
                        sweep_reduce16(q[0], q[1], q[2], q[3], pp_[0], pp_[1], pp_[2], pp_[3], vB[0], vB[1], vB[2], vB[3], vC[0], vC[1], vC[2], vC[3]);
                        *(float2 *)(myQP + r * kCkX + C0) = make_float2(q[0], q[1]);
                        mydB[r * kCkX + C0 + qrow] = vB[0];
                        mydC[r * kCkX + C0 + qrow] = vC[0];
                    } else {
                        group_sum4<NP>(q[0], q[1], q[2], q[3]);
                        group_sum4<NP>(pp_[0], pp_[1], pp_[2], pp_[3]);
                        if (n == 0) {
                            *(float4 *)(sQ + cl * PCH + r * kCkX + C0) = make_float4(q[0], q[1], q[2], q[3]);
                            *(float4 *)(sP + cl * PCH + r * kCkX + C0) = make_float4(pp_[0], pp_[1], pp_[2], pp_[3]);
                        }
                        // sum over the wave's channels: lane bits 4-5 by a swap reduce-scatter (the
                        // 16-lane row q ends with column C0+q), bits 3 and 2 (8- and 4-lane layouts) by row rotates
                        rows_scatter4x2(vB[0], vB[1], vB[2], vB[3], vC[0], vC[1], vC[2], vC[3]);
                        float tb = vB[0], tc = vC[0];
                        if (NP <= 8) { tb += dpp_mov<0x128>(tb); tc += dpp_mov<0x128>(tc); }   // row_ror:8
                        if (NP <= 4) { tb += dpp_mov<0x124>(tb); tc += dpp_mov<0x124>(tc); }   // row_ror:4
                        if ((tid & (16 - NP)) == 0) {
                            mydB[r * kCkX + C0 + qrow] = tb;
                            mydC[r * kCkX + C0 + qrow] = tc;
                        }
                    }
                }
                Gd8 = GR[r];                        // G[r][j0+TE]: diagonal neighbour for the row above
                GR[r] = Gr;                         // G[r][j0]: right neighbour for the tile on the left
                SR[r] = Sr;
                tR[r] = tr;
            }
            GRc = gd_old0;
#pragma unroll
            for (int k = 0; k < NBC; ++k) {         // (ahead of the barrier: behind it another wave may stage the next tile's B and C)
                pB[k] = sB[(wave_u + WPB * k) * NSTR + (tid & 63)];
                pC[k] = sC[(wave_u + WPB * k) * NSTR + (tid & 63)];
            }
            const bool hands_over = PIPE && I == I_lo && I > 0;   // top strip of a band: another block takes the row
            if (!SINGLE && I > 0 && lvalid) {       // adjoint row for the strip above
                char *dst = gdown + (int64_t)J * DN8 * 4;
                if (PIPE) {
#pragma unroll
                    for (int k = 0; k < kCkX; k += 2) st2_coherent((float *)(dst + (k >> 1) * DN2 * 4 + laneG), Gd[k], Gd[k + 1]);
                } else {
                    *(float4 *)(dst + laneG) = make_float4(Gd[0], Gd[1], Gd[2], Gd[3]);
                    *(float4 *)(dst + DN4 * 4 + laneG) = make_float4(Gd[4], Gd[5], Gd[6], Gd[7]);
                }
            }
            __builtin_amdgcn_s_setprio(0);
            if (hands_over) strip_stores_done();
            __syncthreads();
            if (hands_over) strip_signal(progress + I);   // tile J is handed over to the strip above
            // (not ahead of the hand-over: its wait for the row's stores would cover them)
            if (!SINGLE) {
                load_row_ckpt(In, Jn);
                load_col_ckpt(In, Jn);
            }

            Part part;
            flush_read(part);
            __builtin_amdgcn_sched_barrier(0);
            // ---- once per pixel: du, ddelta (thread that staged the pixel), dD, ddelta_bias
            {
            SND_THREAD_MAPS(NP);
            if constexpr (VEC) {
#pragma unroll
                for (int k = 0; k < NCH; ++k) {
                    const int q = n + NP * k;
                    const int row = r0 + (q >> 1), col = j0 + (q & 1) * 4;
                    const float4 q4 = *(const float4 *)(sQ + cl * PCH + q * 4), p4 = *(const float4 *)(sP + cl * PCH + q * 4);
                    const float4 l4 = *(const float4 *)(sDl + cl * DLP + ((q >> 1) + 1) * HG + DLO + (q & 1) * 4);
                    const float4 u4 = *(const float4 *)(sU + cl * PCS + q * 4), o4 = *(const float4 *)(sDo + cl * PCH + q * 4);
                    const float4 g4 = *(const float4 *)(sSg + cl * PCS + q * 4);
                    const float4 ss = *(const float4 *)(sS + q * 4);
                    const float aq[4] = {fmaf(o4.x, ss.x, q4.x), fmaf(o4.y, ss.y, q4.y), fmaf(o4.z, ss.z, q4.z), fmaf(o4.w, ss.w, q4.w)}, ap[4] = {p4.x, p4.y, p4.z, p4.w}, al[4] = {l4.x, l4.y, l4.z, l4.w};
                    const float au[4] = {u4.x, u4.y, u4.z, u4.w}, ao[4] = {o4.x, o4.y, o4.z, o4.w}, ag[4] = {g4.x, g4.y, g4.z, g4.w};
                    float duv[4], ddl[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        duv[e] = fmaf(Dv, ao[e], al[e] * aq[e]);
                        ddl[e] = fmaf(kLn2, ap[e], au[e] * aq[e]) * ag[e];
                    }
                    if (cvalid && row < H && col < W) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            dD_acc = fmaf(ao[e], au[e], dD_acc);
                            dw_acc = fmaf(duv[e], au[e], dw_acc);
                            dbias_acc += ddl[e];
                        }
                        if (fh) {                   // scan order -> memory order
                            const float a0 = duv[0], a1 = duv[1], b0 = ddl[0], b1 = ddl[1];
                            duv[0] = duv[3]; duv[1] = duv[2]; duv[2] = a1; duv[3] = a0;
                            ddl[0] = ddl[3]; ddl[1] = ddl[2]; ddl[2] = b1; ddl[3] = b0;
                        }
                        const uint32_t o = cGb + mad24(mrow(row), WB, mcol(col + (fh ? 3 : 0)) * ESZ);
                        stg4_b(dub, o, duv);
                        stg4_b(ddb, o, ddl);
                    }
                }
            } else {
#pragma unroll
            for (int k = 0; k < NPX; ++k) {
                const int pp = n + NP * k;
                const int row = r0 + (pp >> 3), col = j0 + (pp & 7);
                const float pv = sP[cl * PCH + pp];
                const float dl = sDl[cl * DLP + ((pp >> 3) + 1) * HG + DLO + (pp & 7)];
                const float uv = sU[cl * PCS + pp], dov = sDo[cl * PCH + pp], sg = sSg[cl * PCS + pp];
                const float qv = fmaf(dov, sS[pp], sQ[cl * PCH + pp]);
                const float duv = fmaf(Dv, dov, dl * qv);
                const float ddl = fmaf(kLn2, pv, uv * qv) * sg;
                if (cvalid && (pp >> 3) < TE && (pp & 7) < TE && row < H && col < W) {
                    dD_acc = fmaf(dov, uv, dD_acc);
                    dw_acc = fmaf(duv, uv, dw_acc);
                    dbias_acc += ddl;
                    const uint32_t o = cGb + mad24(mrow(row), WB, mcol(col) * ESZ);
                    stg_b(dub, o, duv);
                    stg_b(ddb, o, ddl);
                }
            }
            }
            }
            flush_bc(part, I, J);
        }
        if (SEG && seg + 1 < geo.nSeg) {
            // hand the carried column state to the block of the strip's next segment: stores, each wave waits for its
            // own to complete, block barrier, then one thread moves the strip's count of finished segments
            float *dst = colstate + (tid << 1);
#pragma unroll
            for (int r = 0; r < kRows; r += 2) {
                st2_coherent(dst + (r >> 1) * 512, GR[r], GR[r + 1]);
                st2_coherent(dst + (4 + (r >> 1)) * 512, SR[r], SR[r + 1]);
                st2_coherent(dst + (8 + (r >> 1)) * 512, tR[r], tR[r + 1]);
            }
            st2_coherent(dst + 12 * 512, GRc, 0.f);
            strip_stores_done();
            __syncthreads();
            strip_signal(segdone + I);
        }
    }
#undef DL
#undef AEXP
#undef EXPA

    // ---- per-lane / per-channel sums leave the kernel
    if (lvalid) glb_add(p.dA + (int64_t)c * N + n, dA_acc);
    dD_acc = group_sum<NP>(dD_acc);
    dbias_acc = group_sum<NP>(dbias_acc);
    if (n == 0 && cvalid) {
        if (p.dD) glb_add(p.dD + c, dD_acc);
        if (p.ddelta_bias) glb_add(p.ddelta_bias + c, dbias_acc);
    }
    if (merge && p.dmerge) {
        dw_acc = group_sum<NP>(dw_acc);
        if (n == 0 && cvalid) glb_add(p.dmerge + c, dw_acc);
    }
    if (p.dA_decay) {
        float v = lvalid ? dec_acc : 0.f;
        v = group_sum<16>(v);
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if ((tid & 63) == 0) sRed[wave] = v;
        __syncthreads();
        if (tid == 0) {
            float t = 0.f;
            for (int w = 0; w < WPB; ++w) t += sRed[w];
            glb_add(p.dA_decay, t / f.A_decay[0]);
        }
    }
}

// Dynamic LDS of one backward block (more than the 64 KB a kernel gets without asking).
template <int NP, int TE> constexpr size_t bwd_lds_bytes() {
    constexpr int PCH = kTile + (NP == 16 ? 8 : 4), PCS = bwd_pcs(NP, TE), NSD = NP == 16 ? kTile + 2 : kTile + 4;
    constexpr int sums = (NP / 4 + 1) * kTile, hold = 2 * NP * kTile;
    return sizeof(float) * (2 * NP * (kTile + 4) + 2 * (NP / 4) * NP * NSD + 16 * 120 + 16 * (3 * PCH + 2 * PCS) + 4 +
                            (TE == 7 ? (hold > sums ? hold : sums) : hold + sums) + NP / 4);
}
// Raise the dynamic LDS limit of every backward instantiation of one input dtype on the current device.
// hipFuncSetAttribute is not stream-ordered and must not run under a stream capture, which is why it is
// done once per device at set-up and not inside the launch path.
template <typename T, int NP, int TE, bool VEC> static bool configure_bwd_one() {
    const int lds = (int)bwd_lds_bytes<NP, TE>();
    if (NP == 16 && hipFuncSetAttribute((const void *)bwd_kernel<T, NP, true, TE, VEC, NP == 16>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
        return false;
    constexpr bool S = TE == 7 || VEC;               // (8x8 tiles element by element: the general kernel)
    if (S && hipFuncSetAttribute((const void *)bwd_kernel<T, NP, false, TE, VEC, false, S>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
        return false;
    return hipFuncSetAttribute((const void *)bwd_kernel<T, NP, true, TE, VEC>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess &&
           hipFuncSetAttribute((const void *)bwd_kernel<T, NP, false, TE, VEC>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
}
template <typename T> int configure_bwd_t() {
    const bool ok = configure_bwd_one<T, 16, 8, false>() && configure_bwd_one<T, 16, 7, false>() && configure_bwd_one<T, 8, 8, false>() &&
                    configure_bwd_one<T, 8, 7, false>() && configure_bwd_one<T, 4, 8, false>() && configure_bwd_one<T, 4, 7, false>() &&
                    configure_bwd_one<T, 16, 8, true>() && configure_bwd_one<T, 8, 8, true>() && configure_bwd_one<T, 4, 8, true>();
    return ok ? SND_OK : SND_ERR_LAUNCH;
}

// Whether a call can stage four columns per access (bwd_kernel's VEC): every row of every tensor the staging touches
// must start on a four-element boundary (16 bytes of fp32, 8 bytes of 16-bit values), and so must the rows of the dense
// du / ddelta; a state's plane of B / C must lie within 2^31 bytes of the first (the state offset is per lane there).
inline bool vec4_ok(const void *ptr, int esz, std::initializer_list<int64_t> strides) {
    if (((uintptr_t)ptr & (uintptr_t)(4 * esz - 1)) != 0) return false;
    for (int64_t s : strides)
        if (s % 4 != 0) return false;
    return true;
}
inline bool bwd_vec_ok(const snd_bwd_params &p) {
    const snd_fwd_params &f = p.f;
    const snd_shape &sh = f.shape;
    const int e = sh.in_dtype == SND_F32 ? 4 : 2, eo = p.dout_dtype == SND_F32 ? 4 : 2;
    if (sh.ncols % 4 != 0) return false;
    const int64_t span = (int64_t)(sh.dstate - 1) * e;
    if (span * f.B_dstate_stride + (int64_t)sh.nrows * f.B_h_stride * e >= ((int64_t)1 << 31) ||
        span * f.C_dstate_stride + (int64_t)sh.nrows * f.C_h_stride * e >= ((int64_t)1 << 31))
        return false;
    return vec4_ok(f.u, e, {f.u_batch_stride, f.u_d_stride, f.u_h_stride}) &&
           vec4_ok(f.delta, e, {f.delta_batch_stride, f.delta_d_stride, f.delta_h_stride}) &&
           vec4_ok(f.B, e, {f.B_batch_stride, f.B_group_stride, f.B_dstate_stride, f.B_h_stride}) &&
           vec4_ok(f.C, e, {f.C_batch_stride, f.C_group_stride, f.C_dstate_stride, f.C_h_stride}) &&
           vec4_ok(p.dout, eo, {p.dout_batch_stride, p.dout_d_stride, p.dout_h_stride}) &&
           vec4_ok(p.du, e, {}) && vec4_ok(p.ddelta, e, {});
}

template <typename T, int NP, int TE, bool VEC>
static int launch_bwd_te(const snd_bwd_params &p, const Geo &geo, hipStream_t stream) {
    const snd_shape &sh = p.f.shape;
    const int rg = sh.dim / sh.n_groups;
    const int nChunks = (rg + 15) / 16;
    const int64_t nPC = (int64_t)sh.batch * sh.n_groups * nChunks;
    constexpr size_t lds = bwd_lds_bytes<NP, TE>();
    const int bands = bwd_band_count(p.f.schedule, (int64_t)sh.batch * sh.n_groups, nChunks, geo.nCY, p.workspace, sh.dstate, geo.nCX);   // 0: one block per plane chunk
    const bool pipe = bands > 0;
    // the dynamic LDS limit of these kernels is raised by snd_init() / on the first launch on a device
    if (int st = ensure_device_ready(); st != SND_OK) return st;
    if (pipe) {
        if (nPC * geo.nCY >= (int64_t)1 << 31) return SND_ERR_SHAPE;
        if (clear_sync_words((int *)p.workspace, sync_words(nPC, geo.nCY), stream) != SND_OK) return SND_ERR_LAUNCH;
        Geo gb = geo;
        gb.spinLimit = spin_limit();
        gb.nBands = bands;
        gb.nQueues = job_queues(sh.batch * sh.n_groups);
        // one strip per job and more strips than block slots: the strips may be cut into column segments (the plan
        // has sized the workspace for their carried state)
        if (bands == geo.nCY && NP == 16) gb.nSeg = strip_segments(nPC, geo.nCY, geo.nCX, bwd_slots(sh.dstate), gb.nQueues);
        gb.segTiles = geo.nCX / gb.nSeg;
        if (nPC * bands * gb.nSeg >= (int64_t)1 << 31) return SND_ERR_SHAPE;
        if (NP == 16 && gb.nSeg > 1)
            hipLaunchKernelGGL((bwd_kernel<T, NP, true, TE, VEC, NP == 16>), dim3((int)(nPC * bands * gb.nSeg)), dim3(16 * NP), lds, stream, p, gb);
        else
            hipLaunchKernelGGL((bwd_kernel<T, NP, true, TE, VEC>), dim3((int)(nPC * bands)), dim3(16 * NP), lds, stream, p, gb);
    } else {
        const int grid = xcd_grid(sh.batch * sh.n_groups, nChunks);
        constexpr bool S = TE == 7 || VEC;
        if (S && geo.nCX == 1 && geo.nCY == 1)
            hipLaunchKernelGGL((bwd_kernel<T, NP, false, TE, VEC, false, S>), dim3(grid), dim3(16 * NP), lds, stream, p, geo);
        else
            hipLaunchKernelGGL((bwd_kernel<T, NP, false, TE, VEC>), dim3(grid), dim3(16 * NP), lds, stream, p, geo);
    }
    return hipGetLastError() == hipSuccess ? SND_OK : SND_ERR_LAUNCH;
}

template <typename T, int NP>
static int launch_bwd_np(const snd_bwd_params &p, hipStream_t stream) {
    Geo geo = make_geo(p.f.shape.nrows, p.f.shape.ncols);
    geo.tag = state_tag(p.f.x_sd, p.f.shape);
    if (geo.te == 7) return launch_bwd_te<T, NP, 7, false>(p, geo, stream);
    return bwd_vec_ok(p) ? launch_bwd_te<T, NP, 8, true>(p, geo, stream) : launch_bwd_te<T, NP, 8, false>(p, geo, stream);
}

// One instantiation per input dtype, each in its own translation unit.
template <typename T>
int launch_bwd_t(const snd_bwd_params &p, hipStream_t stream) {
    const snd_shape &sh = p.f.shape;
    const int N = sh.dstate;
    if (N > 4 && N <= 8) {
        const Geo geo = make_geo(sh.nrows, sh.ncols);
        const int nChunks = (sh.dim / sh.n_groups + 15) / 16;
        const int64_t pairs = (int64_t)sh.batch * sh.n_groups;
        const int jobs = bwd_band_count(p.f.schedule, pairs, nChunks, geo.nCY, p.workspace, N, geo.nCX);
        if (launch_underfilled(pairs * nChunks, jobs, geo.nCY, geo.nCX)) return launch_bwd_np<T, 16>(p, stream);
    }
    return N > 8 ? launch_bwd_np<T, 16>(p, stream) : N > 4 ? launch_bwd_np<T, 8>(p, stream) : launch_bwd_np<T, 4>(p, stream);
}

}  // namespace snd
