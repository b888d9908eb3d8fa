// HIP kernels of the FIP-TOI imaging-and-trigger path for gfx950 (CDNA4).
//
// Per batch of S snapshots the path runs these launches (each covers all S
// snapshots):
//   bin      weighting (FIPkernels.cu:188-195), FP64 uv scaling, each segment of
//            a snapshot's visibilities sorted by grid column; per snapshot the
//            FP64 re-projection geometry and cleared maximum slots
//   merge    a snapshot's segments into one column order (not for one segment)
//   stage1   per uv column c >= 0: deterministic integer LDS gridding of the
//            Hermitian-folded grid column (FIPkernels.cu:197-245) and its
//            length-g inverse FFT along the row axis, cropped to I rows
//   stage2   per two image rows: complex-to-real length-g inverse FFT along the
//            column axis, cropped, |.| and the separable grid correction ->
//            corrected image (FIPkernels.cu:256-287), plus its maximum (spread
//            slots)
//   splat    per target tile: affine + SIN re-projection (FP64 per group of
//            sources, FP32 within it) and the bilinear forward splat
//            accumulated exactly in int32 LDS, plus the image maximum
//            (FIPkernels.cu:289-497)
//   trigger  per tile and window of three images: tLISI (FIPkernels.cu:415-552)
//
// The image identity the stages rely on: with the reference's modulation
// (-1)^(r1+r2) in gridding and the (-1)^(|x|+|y|) flip after the FFT, the
// cropped real part is D[y][x] = Re sum_{r1,r2} Gc[r1][r2] e^{+2 pi i (r1 y + r2 x)/g}
// for the unmodulated grid Gc.  Folding Gc into the Hermitian grid
// Gh[r] = (Gc[r] + conj(Gc[-r]))/2 makes D = sum Gh e^{...} exactly, so only
// columns c = 0..g/2 of Gh are transformed and the second axis is a C2R.
#include "fip_fft.hpp"
#include "fip_internal.hpp"

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <cmath>

namespace fip {

// ---------------------------------------------------------------- helpers

// Spread-slot layout of the image maxima: [S][set 0..1][kMaxSlots] unsigned.
constexpr size_t kPmaxPer = (size_t)2 * kMaxSlots;   // unsigned per snapshot
__host__ __device__ inline size_t max_slot_index(int s, int set, int slot)
{
    return (size_t)s * kPmaxPer + (size_t)set * kMaxSlots + (size_t)slot;
}
__device__ __forceinline__ unsigned* max_slot(unsigned* pm, int s, int set, int slot)
{
    return pm + max_slot_index(s, set, slot);
}
size_t pmax_words(int S) { return (size_t)S * kPmaxPer; }
size_t pmax_index(int s, int set, int slot) { return max_slot_index(s, set, slot); }

template <class T> __device__ __forceinline__ float vis_to_f(const void* p, size_t i);
template <> __device__ __forceinline__ float vis_to_f<float>(const void* p, size_t i)
{
    return static_cast<const float*>(p)[i];
}
template <> __device__ __forceinline__ float vis_to_f<__hip_bfloat16>(const void* p, size_t i)
{
    return __bfloat162float(static_cast<const __hip_bfloat16*>(p)[i]);
}
template <> __device__ __forceinline__ float vis_to_f<__half>(const void* p, size_t i)
{
    return __half2float(static_cast<const __half*>(p)[i]);
}

__device__ __forceinline__ int wave_max_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}
// Max over the 64 lanes (all active), returned in every lane: DPP row shifts
// leave each row of 16 lanes' max in its last lane, and the four row maxima
// are combined as scalars (max is exact in any order).  10 instructions
// instead of 30 for the shuffle butterfly.
__device__ __forceinline__ unsigned wave_max_u(unsigned v)
{
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true));   // row_shr:1
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true));   // row_shr:2
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true));   // row_shr:4
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true));   // row_shr:8
    const unsigned a = (unsigned)__builtin_amdgcn_readlane((int)v, 15);
    const unsigned b = (unsigned)__builtin_amdgcn_readlane((int)v, 31);
    const unsigned c = (unsigned)__builtin_amdgcn_readlane((int)v, 47);
    const unsigned d = (unsigned)__builtin_amdgcn_readlane((int)v, 63);
    return max(max(a, b), max(c, d));
}
// Inclusive sum over the lanes (all active) by DPP: shifts within rows of 16,
// then each row's and each half's total added to the later ones.
__device__ __forceinline__ int wave_scan_i(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
    return v;
}
__device__ __forceinline__ float wave_sum_f(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float wave_max_f(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// Block-wide max of a non-negative float (as ordered bits).  All threads call.
template <int NT>
__device__ __forceinline__ unsigned block_max_u(unsigned v, unsigned* sh)
{
    v = wave_max_u(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    unsigned r = 0;
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < NT / 64; ++i) r = max(r, sh[i]);
    }
    return r;   // valid in thread 0
}

// Workgroups are dispatched round-robin over the 8 XCDs; this maps the
// hardware block id to a logical id so that each XCD works on one contiguous
// run of logical blocks (neighbouring rows/tiles then share an L2).
__device__ __forceinline__ int xcd_remap(int bid, int nb)
{
    constexpr int nx = 8;
    const int per = nb / nx, rem = nb % nx;
    const int x = bid % nx, k = bid / nx;
    return x * per + min(x, rem) + k;
}

// Largest grid size: bounds the keys one scan thread holds.
constexpr int kMaxGrid = 12288;

// ------------------------------------------------------------- front end

// Re-projection geometry of one snapshot from its V matrix (vin, 9 floats).
__device__ SnapGeom snap_geometry(const float* __restrict__ vin, int I, float cell)
{
    // Re-projection geometry (coordschange FIPkernels.cu:289-299 and the
    // closed form of p2p :301-376), FP64 from the float V matrix.
    const float* V = vin;
    const double v00 = V[0], v01 = V[1], v10 = V[3], v11 = V[4];
    const double v20 = V[6], v21 = V[7], v22 = V[8];
    const double a22 = fabs(v22);
    SnapGeom gm;
    gm.m00 = -v00 / a22;
    gm.m01 = v10 / a22;
    gm.m10 = -v01 / a22;
    gm.m11 = v11 / a22;
    const double det = gm.m00 * gm.m11 - gm.m01 * gm.m10;
    gm.i00 = gm.m11 / det;
    gm.i01 = -gm.m01 / det;
    gm.i10 = -gm.m10 / det;
    gm.i11 = gm.m00 / det;
    gm.im00 = fabs(gm.m00) > 1e-12 ? 1.0 / gm.m00 : 0.0;
    gm.im10 = fabs(gm.m10) > 1e-12 ? 1.0 / gm.m10 : 0.0;
    const double xi = v20 / v22, eta = v21 / v22;
    const double delta = (double)cell;
    gm.sx = -xi / delta;
    gm.sy = eta / delta;
    gm.delta = delta;
    gm.sin_on = (xi * xi + eta * eta != 0.0) ? 1 : 0;
    // Singular values of the affine part, and the largest direction-cosine
    // radius any source or target can reach.
    const double h = (double)(I / 2);
    const double tr = gm.m00 * gm.m00 + gm.m01 * gm.m01 + gm.m10 * gm.m10 + gm.m11 * gm.m11;
    const double dd = fabs(det);
    const double disc = sqrt(fmax(0.0, tr * tr - 4.0 * dd * dd));
    const double smax = sqrt(0.5 * (tr + disc)), smin = sqrt(fmax(0.0, 0.5 * (tr - disc)));
    const double rmax = delta * (smax * h * 1.4142135623730951 + 4.0 + h);
    const double kap = sqrt(xi * xi + eta * eta) * rmax / sqrt(fmax(1e-300, 1.0 - rmax * rmax));
    gm.kappa = kap;
    if (!(rmax < 0.9) || !(kap < 0.5) || !isfinite(det) || det == 0.0) {
        gm.curv = -1.0;   // no usable bound: the splat scans whole images
    } else {
        gm.curv = kap;
    }
    // A pixel receives splat weight from the sources mapped into the open
    // 2 x 2 square around it.  The map expands by at least
    // smin (1 - kappa), so they lie in a set of diameter
    // 2 sqrt(2) / (smin (1 - kappa)), which holds at most (d + 1)^2
    // integer points.  Without a usable bound every pixel of the image
    // counts.
    {
        const double den = smin * (1.0 - kap);
        double cap = (gm.curv >= 0.0 && den > 0.0) ? 2.8284271247461903 / den + 1.0 : 0.0;
        cap = cap * cap;
        const double all = (double)I * (double)I;
        gm.ccap = (int)fmin(gm.curv >= 0.0 && den > 0.0 ? ceil(cap) : all, fmin(all, 1073741824.0));
        gm.ccap = max(gm.ccap, 1);
    }
    // n' = 1 - sqrt(1 - r^2) = r^2 (1/2 + r^2/8 + r^4/16 + 5 r^6/128 + ...);
    // for r^2 <= 0.01 the terms after r^8 are below 3e-12 of n'.
    // The splat takes this series along each group of 8 consecutive
    // sources of a row (k = 0..7) from its quadratic Taylor model in k.
    // r^2 is quadratic in k with |dr^2/dk| <= 2 r d and d2r^2/dk2 = 2 d^2,
    // d = cell |(m00, m10)|; for r <= 0.1 the series' third k-derivative
    // is at most 0.31 d^3, so the model's remainder at k <= 7 is at most
    // 17.6 d^3 in n', 17.6 d^3 max(|sx|, |sy|) in pixels.  The series
    // form is taken only where that is at most 5e-8 px (a tenth of an FP32
    // ulp of the splat's local positions); otherwise the closed form per
    // source.
    const double dcol = delta * sqrt(gm.m00 * gm.m00 + gm.m10 * gm.m10);
    const double qerr = 18.0 * dcol * dcol * dcol * fmax(fabs(gm.sx), fabs(gm.sy));
    gm.series = (rmax * rmax <= 0.01 && qerr <= 5e-8) ? 1 : 0;
    gm.pad = 0;
    gm.kratio = kap / (1.0 - kap);
    gm.fm00 = (float)gm.m00;
    gm.fm10 = (float)gm.m10;
    gm.fsx = (float)gm.sx;
    gm.fsy = (float)gm.sy;
    gm.fdelta = (float)gm.delta;
    gm.fdl = -gm.fdelta * gm.fm00;
    gm.fdn = gm.fdelta * gm.fm10;
    gm.padf = 0.0f;
    return gm;
}

// Threads of a bin workgroup.  16 waves each keep the CUs busy although a
// step has at most 64 workgroups per snapshot.
constexpr int kBinThreads = 1024;

// Column keys, in the order of the sorted records.  With the Hermitian fold
// column c takes its own records and the mirrored ones of column -c, so beyond
// the axis b2 = floor(p2) and -b2 share a key, and a column's records are one
// run of keys.  Within eight columns of the axis the sign stays apart
// (0..16 for b2 = -8..8): there a record can reach a column both ways, and a
// column walks its direct and its mirrored run.
__host__ __device__ constexpr int bin_keys(int G) { return G / 2 + 13; }
// Ints of one row of key offsets (keys + 1, in 16-byte units).
__host__ __device__ constexpr int boff_row(int G) { return (bin_keys(G) + 1 + 3) & ~3; }
__device__ __forceinline__ int bin_key(int b2) { return 8 + (b2 < -8 ? -b2 : b2); }

// Grid coordinates and weighted value of one visibility as a record, and its
// column key; -1 where it has no tap.  rj = 1 / |V00 V11 - V01 V10|
// (computeVisWeighted, FIPkernels.cu:188-195); positions in FP64, B * (cell g)
// (FIPkernels.cu:211-212, 584).  r1, r2: largest |tap| on each axis.
__device__ __forceinline__ int vis_record(float vr, float vi, float b1, float b2, double rj, double scale, int G,
                                          VisRec& r, int& r1, int& r2)
{
    const int M = G / 2;
    const double p1 = (double)b1 * scale, p2 = (double)b2 * scale;
    // Coordinates far outside the grid have no taps (and must not overflow int).
    if (!(fabs(p1) < (double)G && fabs(p2) < (double)G)) return -1;
    const double fb1 = floor(p1), fb2 = floor(p2);
    const float f1 = (float)(p1 - fb1), f2 = (float)(p2 - fb2);
    const int i1 = (int)fb1, i2 = (int)fb2;
    // Taps: r in [ceil(p-4), floor(p+4)] (FIPkernels.cu:213-243), eight, or
    // nine where the position is an integer.
    const int nine1 = f1 > 0.0f ? 0 : 1, nine2 = f2 > 0.0f ? 0 : 1;
    const int lo1 = i1 - 3 - nine1, hi1 = i1 + 4, lo2 = i2 - 3 - nine2, hi2 = i2 + 4;
    const int clo1 = max(lo1, -M), chi1 = min(hi1, M - 1), clo2 = max(lo2, -M), chi2 = min(hi2, M - 1);
    if (clo1 > chi1 || clo2 > chi2) return -1;
    const int edge = (lo1 <= -M || hi1 >= M) ? 1 : 0;
    r.row = (lo1 << 2) | (nine1 << 1) | edge;
    r.f1 = nine1 ? 1.0f : f1;
    r.col = (lo2 << 1) | nine2;
    r.f2 = nine2 ? 1.0f : f2;
    r.vr = (float)((double)vr * rj);
    r.vi = (float)((double)vi * rj);
    r1 = max(chi1, -clo1);
    r2 = max(chi2, -clo2);
    return bin_key(i2);
}

// Field k of a snapshot's gridded extent: largest |column tap|, |row tap| and
// weighted magnitude (float bits).
__device__ __forceinline__ void set_extent(SnapMeta& m, int k, int v)
{
    if (k == 0) m.rmax = v;
    if (k == 1) m.r1max = v;
    if (k == 2) m.maxv_bits = (unsigned)v;
}

// One segment of one snapshot's visibilities into column order: records and
// keys, an LDS histogram whose atomics give each record its place within its
// key, the exclusive scan of the counts, and the records to their places in
// the segment's own stretch of the output, with the segment's key offsets.
// Nothing is combined across workgroups here: no zeroed counters and no
// global atomics.  A snapshot of one segment is done with that; k_merge puts
// several into one order.
//
// VPT visibilities per thread held in registers between the two phases; 0:
// any number, recomputed in the second phase.  Workgroup `nseg` of a snapshot
// sets up what the later stages need: geometry, normalisation and cleared
// maximum slots.
//
// Latency bound: at 2048^2 with 32640 visibilities 1.2 us of loads, 1.7 of
// FP64 and LDS atomics, 1.5 of scan and 0.6 of stores; the rest of its 8 us is
// launch and write-back.  With k_merge 7, 14, 16, 25 and 59 us (rocprofv3, three
// snapshots) at 256^2, 1024^2, 2048^2, 4096^2 and 8192^2 with 2016, 8128, 32640,
// 130816 and 523776 visibilities (the last two with k_offsets); clearing,
// histogram with global atomics, scan and scatter as four launches took 16, 18,
// 21, 32 and 73.  (A column
// kernel that took its records from the sorted segments themselves, with no
// merge, lost more than the merge costs: 95 against 84 us at 4096^2.)
template <class VT, int VPT>
__global__ __launch_bounds__(kBinThreads) void k_bin(InputView in, BinView out, const int* __restrict__ norm_n,
                                                     int norm_const, int G, int I, float cell, double scale)
{
    extern __shared__ int lh[];   // bin_keys(G) + 1 ints: counts, then starts
    constexpr int NW = kBinThreads / 64;
    constexpr int PER = (bin_keys(kMaxGrid) + kBinThreads - 1) / kBinThreads;   // keys per thread of the scan
    __shared__ int sh_i[3][NW];
    const int s = blockIdx.y, seg = blockIdx.x, t = threadIdx.x, lane = t & 63, wid = t >> 6;
    const float* V = in.vin + (size_t)s * 9;
    if (seg == out.nseg) {
        if (t < 2 * kMaxSlots) *max_slot(out.pmax, s, 0, t) = 0u;
        if (t == 128) out.geom[s] = snap_geometry(V, I, cell);
        if (t == 192) {
            out.meta[s].maxp_bits = 0u;
            out.meta[s].maxd_bits = 0u;
            out.meta[s].norm_n = norm_n ? norm_n[s] : norm_const;
        }
        return;
    }
    const int ns = in.nvis ? in.nvis[s] : in.n_const;
    const int K = bin_keys(G);
    const int beg = seg * out.chunk, end = min(beg + out.chunk, ns);
    const double rj = 1.0 / fabs((double)V[0] * (double)V[4] - (double)V[1] * (double)V[3]);
    const size_t sbase = (size_t)s * in.stride;
    int rmax = -1, r1max = -1;
    unsigned vmax = 0u;
    VisRec rec[VPT > 0 ? VPT : 1];
    int key[VPT > 0 ? VPT : 1], slot[VPT > 0 ? VPT : 1];
    auto note = [&](const VisRec& r, int r1, int r2) {
        rmax = max(rmax, r2);
        r1max = max(r1max, r1);
        vmax = max(vmax, __float_as_uint(fmaxf(fabsf(r.vr), fabsf(r.vi))));
    };
    // Every input of the thread's visibilities is loaded before any is used,
    // so the loads are in flight together: unconditionally, from an index
    // clamped into this snapshot's rows (entries past its count are loaded
    // but not used), since a load behind a per-lane test would wait in turn.
    float lvr[VPT > 0 ? VPT : 1], lvi[VPT > 0 ? VPT : 1], lb1[VPT > 0 ? VPT : 1], lb2[VPT > 0 ? VPT : 1];
    auto load = [&](int k, int n) {
        const size_t q = sbase + (size_t)n;
        lvr[k] = vis_to_f<VT>(in.vis_re, q);
        lvi[k] = vis_to_f<VT>(in.vis_im, q);
        lb1[k] = in.bin[2 * q];
        lb2[k] = in.bin[2 * q + 1];
    };
    if constexpr (VPT > 0) {
        if (beg < end) {
#pragma unroll
            for (int k = 0; k < VPT; ++k) load(k, min(beg + k * kBinThreads + t, end - 1));
        }
    }
    for (int b = t; b <= K; b += kBinThreads) lh[b] = 0;
    __syncthreads();
    if constexpr (VPT > 0) {
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            int r1, r2;
            key[k] = beg + k * kBinThreads + t < end
                         ? vis_record(lvr[k], lvi[k], lb1[k], lb2[k], rj, scale, G, rec[k], r1, r2)
                         : -1;
            if (key[k] >= 0) {
                slot[k] = atomicAdd(&lh[key[k]], 1);
                note(rec[k], r1, r2);
            }
        }
    } else {
        for (int n = beg + t; n < end; n += kBinThreads) {
            int r1, r2;
            load(0, n);
            const int b = vis_record(lvr[0], lvi[0], lb1[0], lb2[0], rj, scale, G, rec[0], r1, r2);
            if (b >= 0) {
                atomicAdd(&lh[b], 1);
                note(rec[0], r1, r2);
            }
        }
    }
    rmax = wave_max_i(rmax);
    r1max = wave_max_i(r1max);
    vmax = wave_max_u(vmax);
    if (lane == 0) {
        sh_i[0][wid] = rmax;
        sh_i[1][wid] = r1max;
        sh_i[2][wid] = (int)vmax;
    }
    __syncthreads();
    if (t < 3) {   // the float bits of a non-negative maximum order as int
        int v = sh_i[t][0];
        for (int k = 1; k < NW; ++k) v = max(v, sh_i[t][k]);
        if (out.nseg > 1)
            out.seg[(size_t)s * out.seg_stride + t * kMaxSegs + seg] = v;
        else
            set_extent(out.meta[s], t, v);
    }
    // Exclusive scan: each thread's run of keys in registers, shuffles within
    // a wave, the wave totals summed by everyone.
    const int per = (K + kBinThreads - 1) / kBinThreads;
    int v[PER], local = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int b = t * per + k;
        v[k] = (k < per && b < K) ? lh[b] : 0;
        local += v[k];
    }
    int x = local;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    __syncthreads();   // sh_i is read, the counts are in registers
    if (lane == 63) sh_i[0][wid] = x;
    __syncthreads();
    int run = x - local;
#pragma unroll
    for (int k = 0; k < NW; ++k) run += k < wid ? sh_i[0][k] : 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int b = t * per + k;
        if (k < per && b < K) lh[b] = run;
        run += v[k];
    }
    if (t == kBinThreads - 1) lh[K] = run;
    __syncthreads();
    int* o = out.nseg > 1 ? out.boff + (size_t)s * out.boff_stride + (size_t)seg * boff_row(G)
                          : out.bstart + (size_t)s * boff_row(G);
    for (int b = t; b <= K; b += kBinThreads) o[b] = lh[b];
    VisRec* dst = (out.nseg > 1 ? out.rec : out.sorted) + sbase + (size_t)beg;
    if constexpr (VPT > 0) {
#pragma unroll
        for (int k = 0; k < VPT; ++k)
            if (key[k] >= 0) dst[lh[key[k]] + slot[k]] = rec[k];
    } else {
        __syncthreads();   // the offsets are stored; the starts become cursors
        for (int n = beg + t; n < end; n += kBinThreads) {
            int r1, r2;
            load(0, n);
            const int b = vis_record(lvr[0], lvi[0], lb1[0], lb2[0], rj, scale, G, rec[0], r1, r2);
            if (b >= 0) dst[atomicAdd(&lh[b], 1)] = rec[0];
        }
    }
}

// Sum of rows [lo, hi) of four neighbouring keys' offsets, sixteen loads in
// flight (rows past the end are read as the last one and masked off).
__device__ __forceinline__ int4 sum_rows(const int* __restrict__ o, int row, int lo, int hi)
{
    int4 sum = make_int4(0, 0, 0, 0);
    for (int g0 = lo; g0 < hi; g0 += 16) {
        int4 x[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) x[k] = *reinterpret_cast<const int4*>(o + (size_t)min(g0 + k, hi - 1) * row);
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int m = g0 + k < hi ? -1 : 0;
            sum.x += x[k].x & m;
            sum.y += x[k].y & m;
            sum.z += x[k].z & m;
            sum.w += x[k].w & m;
        }
    }
    return sum;
}

// Where many segments' records go: workgroups of 64 keys by 16 groups of
// segments add boff up once and store the displacement of every segment's
// records of a key (see k_merge), and the snapshot's offsets.
__global__ __launch_bounds__(1024) void k_offsets(BinView v, int G)
{
    constexpr int GR = 16, PER = kMaxSegs / GR;
    static_assert(kMaxSegs % GR == 0, "whole groups");
    __shared__ int part[GR][2][64];
    const int s = blockIdx.y, lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int K = bin_keys(G), row = boff_row(G);
    const int k = blockIdx.x * 64 + lane, ka = min(k, K), kb = min(k + 1, K);
    const int* bo = v.boff + (size_t)s * v.boff_stride;
    int a[PER], b[PER], sa = 0, sb = 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) {   // segments past the end are read as the last one and masked off
        const int g = grp * PER + q, m = g < v.nseg ? -1 : 0;
        const int* o = bo + (size_t)min(g, v.nseg - 1) * row;
        a[q] = o[ka] & m;
        b[q] = o[kb] & m;
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        sa += a[q];
        sb += b[q];
    }
    part[grp][0][lane] = sa;
    part[grp][1][lane] = sb;
    __syncthreads();
    int after = 0, before = 0, total = 0;   // of this key in this group's and later, of the next in earlier segments
#pragma unroll
    for (int e = 0; e < GR; ++e) {
        const int x = part[e][0][lane];
        total += x;
        after += e < grp ? 0 : x;
        before += e < grp ? part[e][1][lane] : 0;
    }
    if (grp == 0 && k <= K) v.bstart[(size_t)s * row + k] = total;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int g = grp * PER + q;
        after -= a[q];
        if (g < v.nseg && k < K) v.disp[(size_t)s * v.seg_stride + (size_t)g * row + k] = after + before;
        before += b[q];
    }
}

// A snapshot's segments into one column order.  boff[g] is segment g's own
// exclusive scan, so the scan of the whole snapshot is its sum over the
// segments, and a record of segment `seg` and key k moves up by the later
// segments' offsets of k (what they hold before k) and the earlier segments'
// offsets of k + 1 (what they hold up to k).  Of few segments every workgroup
// adds the rows of offsets up by itself (four keys per load, from L2) rather
// than wait for a launch that does, and segment 0's also writes the snapshot's
// offsets; SUMMED: k_offsets has.  Segment 0 writes the snapshot's extent.
template <bool SUMMED>
__global__ __launch_bounds__(kBinThreads) void k_merge(BinView v, int G)
{
    extern __shared__ int lds[];   // boff_row(G) ints, twice unless SUMMED
    const int s = blockIdx.y, seg = blockIdx.x, t = threadIdx.x;
    const int K = bin_keys(G), row = boff_row(G);
    int* before = lds;
    int* after = lds + row;
    const int* bo = v.boff + (size_t)s * v.boff_stride;
    const int cnt = bo[(size_t)seg * row + K];
    const VisRec* src = v.rec + (size_t)s * v.stride + (size_t)seg * v.chunk;
    VisRec* dst = v.sorted + (size_t)s * v.stride;
    auto put = [&](VisRec q, int i) {
        const int key = bin_key((q.col >> 1) + 3 + (q.col & 1));
        dst[i + (SUMMED ? before[key] : after[key] + before[key + 1])] = q;
    };
    // The first records are loaded before their displacement is known (the
    // segment has at least one place).
    const int last = max(cnt - 1, 0);
    const VisRec r0 = src[min(t, last)], r1 = src[min(t + kBinThreads, last)];
    for (int b = 4 * t; b < row; b += 4 * kBinThreads) {
        if constexpr (SUMMED) {
            *reinterpret_cast<int4*>(before + b) = *reinterpret_cast<const int4*>(
                v.disp + (size_t)s * v.seg_stride + (size_t)seg * row + b);
            continue;
        }
        const int4 lo = sum_rows(bo + b, row, 0, seg), hi = sum_rows(bo + b, row, seg + 1, v.nseg);
        *reinterpret_cast<int4*>(before + b) = lo;
        *reinterpret_cast<int4*>(after + b) = hi;
        if (seg == 0) {
            const int4 own = *reinterpret_cast<const int4*>(bo + b);
            *reinterpret_cast<int4*>(v.bstart + (size_t)s * row + b) =
                make_int4(own.x + hi.x, own.y + hi.y, own.z + hi.z, own.w + hi.w);
        }
    }
    if (seg == 0 && t < 64) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int* sm = v.seg + (size_t)s * v.seg_stride + k * kMaxSegs;
            const int m = wave_max_i(t < v.nseg ? sm[t] : -1);
            if (t == 0) set_extent(v.meta[s], k, m);
        }
    }
    __syncthreads();
    if (t < cnt) put(r0, t);
    if (t + kBinThreads < cnt) put(r1, t + kBinThreads);
    for (int i = t + 2 * kBinThreads; i < cnt; i += kBinThreads) put(src[i], i);
}

// ---------------------------------------------------------------- stage 1

// One visibility record prepared for a column.  The column weight
// ES((col - p2)/4)/2 (the Hermitian fold's 1/2) is folded into its value.
// Rows are counted from -g/2 (u = row + g/2); taps in ascending u: the first
// row u0 and the tap distances X_j = j - 3 - f, j = 0..7 (and j = 8 where the
// position is an integer: f = 1).  A mirrored record contributes conj(v) at
// row -r, whose taps are those of the position -p1: f = 1 - frac.  A record
// whose taps reach the grid's edge is marked (edge): its taps are clipped and
// a mirrored tap at -g/2 stays there, so each one is placed by itself.
struct ColRec {
    int lo1, u0;
    float f, vr, vi;
    int nine;
    bool mirror, edge, live;
};

// exp(beta*(sqrt(1-x^2)-1)) (FIPkernels.cu:67-71) of a tap distance X = 4x in
// cells, |X| <= 4, as 2^(C s - C) with C = beta log2 e and s = sqrt(1 - x^2)
// (1 - x^2 by one FMA, hardware sqrt and exp2, ~1 ulp each; the 1/16 of X^2
// is moved into the constants, powers of two).  s <= 1 carries an absolute
// error of ~1e-7, so the exponent's error stays below ~2e-6 (C = 22.2) and
// the relative error of ES below ~1.5e-6 at every x.  The form without the
// subtraction, exp(-beta x^2 / (1 + s)), is no more accurate at this precision
// and costs a reciprocal and three more instructions per tap.
__device__ __forceinline__ float es_tap(float X)
{
    constexpr float C = (float)(kBeta * 1.4426950408889634);
    return __builtin_amdgcn_exp2f(fmaf(0.25f * C, __builtin_amdgcn_sqrtf(fmaf(-X, X, 16.0f)), -C));
}

__device__ __forceinline__ ColRec prep_rec(const VisRec& r, int col, bool mirror, int M)
{
    ColRec c;
    c.lo1 = r.row >> 2;
    c.nine = (r.row >> 1) & 1;
    c.edge = r.row & 1;
    c.mirror = mirror;
    c.f = mirror && !c.nine ? 1.0f - r.f1 : r.f1;
    c.u0 = mirror ? M - (c.lo1 + 7 + c.nine) : M + c.lo1;
    const int d = col - (r.col >> 1);   // the column's place among the record's taps
    c.live = (unsigned)d <= (unsigned)(7 + (r.col & 1));
    const float w2 = es_tap((float)(d - 3) - r.f2) * 0.5f;   // only of a live record
    c.vr = r.vr * w2;
    c.vi = (mirror ? -r.vi : r.vi) * w2;
    return c;
}

// floor(x) and floor(x + 0.5) as int32 in one instruction each (the compiler
// keeps floor and the conversion separate without finite-math flags).
__device__ __forceinline__ int cvt_floor_i32(float x)
{
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}
__device__ __forceinline__ int cvt_round_half_up_i32(float x)
{
    int r;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// Shape of the column kernel.  Rows are grouped in blocks of RBS rows, each
// with its own power-of-two scale: at least 16 rows, so that the nine taps of
// a record reach at most two blocks, and at most 96 blocks.
//
// NC copies of the int32 column spread the taps that several lanes of a wave
// put on one row (the uv coverage is dense at the centre: a fifth of a hot
// column's records share one cell at 256^2) over NC addresses; the sums are
// integers, so adding the copies up is exact.  As many copies as keep the
// column under 25 KB.
//
// NX threads are launched and the FFT takes the first NT.  A column with more
// than two records per FFT thread is gridded by as many waves as give each
// thread two (the uv coverage is concentrated: at 2048^2 with 32640
// visibilities the median column holds 118 records and the fullest 4152, and
// with 256 threads that one workgroup ran 33 us, the whole launch); the other
// waves end at once and free their slots.  Where the FFT itself takes 512
// threads or more the launch has workgroups enough to hide the full columns,
// and waves that only end would halve the workgroups per CU.
template <int G>
struct ColShape {
    static constexpr int M = G / 2, I = 2 * G / 3, h = I / 2;
    static constexpr int NT = FftPlan<G>::nt;
    static constexpr int NX = G <= 96 ? 512 : (G <= 1536 ? 1024 : (NT < 512 ? 512 : NT));
    static constexpr int RBS = (G / 96 > 16) ? G / 96 : 16;
    static constexpr int NBLK = G / RBS;
    static constexpr int NC = G <= 384 ? 8 : (G <= 768 ? 4 : (G <= 1536 ? 2 : 1));
    static constexpr int MC = 16;   // copies of a block's mass
    // Waves per SIMD the registers must leave room for: what the LDS allows
    // (three workgroups per CU at g = 6144, one at 12288).
    static constexpr int waves = G >= 12288 ? 4 : (G >= 6144 ? 6 : 2);
    static constexpr int acc_bytes = 2 * G * NC * (int)sizeof(int);
    static constexpr int fft_bytes = lds_len(G) * (int)sizeof(float2);
    static constexpr int bytes = acc_bytes > fft_bytes ? acc_bytes : fft_bytes;
    static constexpr int mass_bytes = NBLK * MC * (int)sizeof(unsigned long long);
    static_assert(G % RBS == 0 && M % RBS == 0 && NBLK <= 96, "scale blocks");
    static_assert(mass_bytes <= acc_bytes && acc_bytes % 16 == 0 && mass_bytes % 16 == 0, "mass inside the column");
    static_assert(NT <= NX && NBLK <= NT * 2, "one round of block scales");
};

// Row taps of one prepared record, accumulated as integers into the LDS
// column (re [0, G), im [G, 2G), each row NC copies; this lane's copy), each
// scaled by its block's power of two and rounded half up.  Away from the
// grid's edge a record's rows are one run u0..u0+7 (u0+8), so every tap is
// one LDS address plus a constant.  It reaches at most two scale blocks, both
// read once: taps from row `cross` on take the second.
template <int G>
__device__ __forceinline__ void grid_taps(const ColRec& c, const float* sc, int* col)
{
    using Sh = ColShape<G>;
    constexpr int NC = Sh::NC, M = Sh::M;
    const int cp = NC > 1 ? (int)(threadIdx.x & (NC - 1)) : 0;
    if (!c.edge) {
        const unsigned ba = (unsigned)c.u0 / (unsigned)Sh::RBS, bz = (unsigned)(c.u0 + 8) / (unsigned)Sh::RBS;
        const float sca = sc[ba], scz = sc[min(bz, (unsigned)Sh::NBLK - 1)];
        const int cross = (int)((ba + 1) * (unsigned)Sh::RBS) - c.u0;
        int* p = col + c.u0 * NC + cp;
        auto tap = [&](int j) {
            const float X = (float)(j - 3) - c.f;
            const float wk = es_tap(X) * (j < cross ? sca : scz);
            atomicAdd(p + j * NC, cvt_round_half_up_i32(c.vr * wk));
            atomicAdd(p + (G + j) * NC, cvt_round_half_up_i32(c.vi * wk));
        };
#pragma unroll
        for (int j = 0; j < 8; ++j) tap(j);
        if (c.nine) tap(8);
        return;
    }
    for (int j = 0; j < 8 + c.nine; ++j) {
        const int t1 = c.mirror ? c.lo1 + 7 + c.nine - j : c.lo1 + j;   // the record's own row
        if (t1 < -M || t1 > M - 1) continue;
        const int u = (c.mirror ? (t1 == -M ? -M : -t1) : t1) + M;
        const float wk = es_tap((float)(j - 3) - c.f) * sc[u / Sh::RBS];
        atomicAdd(col + u * NC + cp, cvt_round_half_up_i32(c.vr * wk));
        atomicAdd(col + (G + u) * NC + cp, cvt_round_half_up_i32(c.vi * wk));
    }
}

// Adds the record's magnitude bound (units of amax / 4096, rounded up) to the
// mass of every scale block its taps touch (at most two).  The mass is 64-bit:
// a column holds up to two records per visibility (its direct and mirrored
// runs), so a 32-bit sum of up to 4096 units per record would wrap after
// about 2^19 visibilities at one uv point.  Each block's mass is kept in MC
// copies, one per lane modulo MC: nearly all records of a full column lie in
// the few blocks around row 0, where a single word per block would serialise
// the wave.
template <int G>
__device__ __forceinline__ void tap_mass(const ColRec& c, float qs, unsigned long long* mass)
{
    using Sh = ColShape<G>;
    const unsigned long long q = (unsigned long long)ceilf(fmaxf(fabsf(c.vr), fabsf(c.vi)) * qs);
    int ba, bz;
    if (!c.edge) {
        ba = c.u0 / Sh::RBS;
        bz = (c.u0 + 7 + c.nine) / Sh::RBS;
    } else {
        const int lo1 = max(c.lo1, -Sh::M), hi1 = min(c.lo1 + 7 + c.nine, Sh::M - 1);
        const int a = c.mirror ? (lo1 == -Sh::M ? -Sh::M : -lo1) : lo1;
        ba = (a + Sh::M) / Sh::RBS;
        bz = ((c.mirror ? (hi1 == -Sh::M ? -Sh::M : -hi1) : hi1) + Sh::M) / Sh::RBS;
        // a clipped mirrored run that starts at -g/2 goes on at the other end
        if (c.mirror && lo1 == -Sh::M && hi1 > lo1) {
            const int bn = (-(lo1 + 1) + Sh::M) / Sh::RBS;
            if (bn != bz) atomicAdd(&mass[bn * Sh::MC + (threadIdx.x & (Sh::MC - 1))], q);
        }
    }
    atomicAdd(&mass[ba * Sh::MC + (threadIdx.x & (Sh::MC - 1))], q);
    if (bz != ba) atomicAdd(&mass[bz * Sh::MC + (threadIdx.x & (Sh::MC - 1))], q);
}

// Runs of the sorted records that can reach column c: [x, y) and [z, w).  The
// first holds column c's own records, beyond eight columns from the axis with
// the mirrored ones of column -c among them; nearer the axis those are the
// second run.  Column g/2 is its own mirror and walks its records both ways.
template <int G>
__device__ __forceinline__ int4 column_ranges(const int* __restrict__ bst, int c)
{
    constexpr int M = G / 2, K = bin_keys(G);
    const int a0 = c + 4, a1 = min(c + 12, K - 1);
    const int b0 = c <= 4 ? 4 - c : 0, b1 = 12 - c;
    int4 r;
    r.x = bst[a0];
    r.y = bst[a1 + 1];
    r.z = c == M ? r.x : (c <= 12 ? bst[b0] : 0);
    r.w = c == M ? r.y : (c <= 12 ? bst[b1 + 1] : 0);
    return r;
}

// Grids column c of snapshot s into LDS, transforms it and stores its I
// cropped rows.  Bound by VALU issue at 4096^2 (the FFT is two thirds of its
// instructions) and by the fullest columns' passes up to 2048^2.  Rows
// counted from -g/2, so that a record's taps are one address plus constants,
// the transform reading the integers and storing the crop from registers, and
// extra waves for full columns took it from 97 to 76 us (4096^2, 130816
// visibilities), 35 to 25 us (2048^2, 32640), 539 to 459 us (8192^2, 523776)
// and 12.4 to 7.6 us (256^2, 2016) for three snapshots (rocprofv3).
//
// smem: ColShape<G>::bytes of LDS, used in turn as the blocks' masses, the int32
// column and the FFT's exchange buffer.  KR records per thread are held in
// registers at a time.
template <int G, int KR>
__device__ __forceinline__ void stage1_column(int s, int c, int4 rg, const VisRec* __restrict__ sorted,
                                              const SnapMeta& m, const float2* __restrict__ tw,
                                              float2* __restrict__ kt, size_t stride, unsigned char* smem, float* sc,
                                              float* isc)
{
    using Sh = ColShape<G>;
    constexpr int NT = Sh::NT, M = Sh::M, RBS = Sh::RBS, NC = Sh::NC;
    const int t = threadIdx.x;

    const VisRec* vs = sorted + (size_t)s * stride;
    const int cc = (c == M) ? -M : c;                        // direct column (centred)
    const int cm = (c == 0) ? 0 : ((c == M) ? -M : -c);      // mirrored column
    const int d0 = rg.x, d1 = rg.y, m0 = rg.z, m1 = rg.w;
    const int nd = d1 - d0, ntot = nd + (m1 - m0);
    const bool by_run = c <= 4 || c == M;   // direct or mirrored by the run it is in, else by its side
    // Threads that grid (whole waves; every condition on them is uniform).
    const int na = min(max((ntot / KR + 63) & ~63, NT), Sh::NX);
    if (t >= na) return;

    // Exact integer accumulation with one power-of-two scale per block of
    // rows.  Pass 1 adds, per block, an upper bound of the magnitudes of the
    // records whose taps reach it (integers, so the bound does not depend on
    // the order of the LDS atomics); the scale keeps every int32 cell sum of
    // the block below 2^29 in magnitude.  Pass 2 accumulates the scaled,
    // rounded contributions; sums of integers are exact, so the column does
    // not depend on the order of the atomics either.
    const float maxv = __uint_as_float(m.maxv_bits);
    const float amax = fmaxf(0.5f * maxv, 1e-30f);   // |v| ES / 2 <= amax
    const float qs = 4096.0f / amax;

    // The two runs in one numbering.  A column whose records do not fit the
    // registers walks them in passes, the next pass's records loaded under
    // this one's work.
    const int step = KR * na;
    VisRec rn[KR];
    ColRec cr[KR];
    auto fetch = [&](int base) {
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const int n = base + k * na + t;
            if (n < ntot) rn[k] = vs[n < nd ? d0 + n : m0 + (n - nd)];
        }
    };
    auto prep = [&](int base) {
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const int n = base + k * na + t;
            if (n < ntot) {
                const bool mirror = by_run ? n >= nd : (rn[k].col >> 1) + (rn[k].col & 1) < -3;   // b2 < 0
                cr[k] = prep_rec(rn[k], mirror ? cm : cc, mirror, M);
            } else {
                cr[k].live = false;
            }
        }
    };
    const bool resident = ntot <= step;
    fetch(0);
    unsigned long long* mass = reinterpret_cast<unsigned long long*>(smem);
    int* col = reinterpret_cast<int*>(smem);
    {
        int4* z = reinterpret_cast<int4*>(smem);
        for (int i = t; i < Sh::acc_bytes / 16; i += na) z[i] = make_int4(0, 0, 0, 0);
    }
    __syncthreads();
    for (int base = 0; base < ntot; base += step) {
        prep(base);
        if (base + step < ntot) fetch(base + step);
#pragma unroll
        for (int k = 0; k < KR; ++k)
            if (cr[k].live) tap_mass<G>(cr[k], qs, mass);
    }
    if (!resident) fetch(0);
    __syncthreads();
    for (int i = t; i < Sh::NBLK; i += na) {
        // One thread per block adds the copies up (starting at its own bank)
        // and leaves them zero for the column that shares their memory.
        unsigned long long sum = 0ull;
#pragma unroll
        for (int k = 0; k < Sh::MC; ++k) {
            unsigned long long* q = mass + i * Sh::MC + ((k + i) & (Sh::MC - 1));
            sum += *q;
            *q = 0ull;
        }
        // bound = mass * amax / 4096 (+ one unit per record of rounding slack
        // is already inside the ceil); 2^e > bound.
        const float bound = (float)sum * (amax / 4096.0f) * 1.0001f;
        int e = 0;
        frexpf(fmaxf(bound, 1e-30f), &e);
        const int k = min(29 - e, 120);   // empty blocks: any finite scale
        sc[i] = ldexpf(1.0f, k);
        isc[i] = ldexpf(1.0f, -k);
    }
    __syncthreads();
    for (int base = 0; base < ntot; base += step) {
        if (!resident) {
            prep(base);
            if (base + step < ntot) fetch(base + step);
        }
#pragma unroll
        for (int k = 0; k < KR; ++k)
            if (cr[k].live) grid_taps<G>(cr[k], sc, col);
    }
    __syncthreads();
    if (t >= NT) return;
    // Column FFT straight from the integer column: element n of the transform
    // is grid row n (n < g/2) or n - g, i.e. u = (n + g/2) mod g, so a
    // butterfly's inputs lie N/R apart here too.
    //
    // Crop y in [-h, h): outputs n < h are rows n, n >= g - h rows n - g, and
    // with the last radix a multiple of 3 and h = g/3 those are whole
    // outputs of each butterfly, stored from its registers.  The row
    // correction 1/(c(|y|) norm) is a factor per image row, applied by the
    // row pass (one load per row there instead of one per row and column
    // here).
    constexpr int R0 = FftPlan<G>::radix[0], NB0 = G / R0;
    constexpr int R1 = FftPlan<G>::radix[FftPlan<G>::nstages - 1], NS1 = G / R1;
    static_assert(R0 % 2 == 0 && R1 % 3 == 0 && NS1 % kKTile == 0 && Sh::h % kKTile == 0, "column plan");
    float2* fb = reinterpret_cast<float2*>(smem);
    float2* ks = kt + (size_t)s * ((size_t)Sh::I * (M + 1)) + (size_t)c * kKTile;
    // NZ: inputs 0..NZ-1 and R0-NZ..R0-1 are read, rows |r| < NZ NB0.
    auto transform = [&](auto NZ) {
        constexpr int nz = decltype(NZ)::value;
        constexpr unsigned mask = band_mask<R0, nz, nz>();
        fft_inverse_io<G, true, false, mask>(
            fb, tw, t,
            [&](int j, int r) {
                const int q0 = NB0 * ((r + R0 / 2) % R0), u = j + q0;
                int re = 0, im = 0;
#pragma unroll
                for (int q = 0; q < NC; ++q) {
                    re += col[u * NC + q];
                    im += col[(G + u) * NC + q];
                }
                const float k = NB0 % RBS == 0 ? isc[j / RBS + q0 / RBS] : isc[u / RBS];
                float2 x = make_float2((float)re * k, (float)im * k);
                // Scaled here, not in the radix-32 butterfly's own multiply-adds:
                // those kept the scales in registers and spilled.
                if constexpr (R0 == 32) asm("" : "+v"(x.x), "+v"(x.y));
                return x;
            },
            [&](int j, const float2* v) {
                float2* o = ks + (size_t)(j / kKTile) * (M + 1) * kKTile + (j % kKTile);
#pragma unroll
                for (int r = 0; r < R1; ++r) {
                    if (r >= R1 / 3 && r < 2 * R1 / 3) continue;
                    const int yp = r < R1 / 3 ? NS1 * r + Sh::h : NS1 * r - G + Sh::h;   // plus j
                    o[(size_t)(yp / kKTile) * (M + 1) * kKTile] = v[r];
                }
            });
    };
    // Rows beyond +-r1max hold no tap, and butterflies drop inputs known to be
    // zero.  The one pruned form takes 9/32 of the first radix's inputs at
    // either end, rounded up: taps below 9/32 of the grid with radix 32 first
    // (4096^2), below 5/16 with radix 16; radix 8 (64^2, 256^2) has none.  It
    // covers baselines up to 0.28 of the sampling rate (3.6 pixels to a period of
    // the longest one's fringe); wider coverage, up to 0.5, takes the full
    // transform.  A call of three snapshots of 130816 at 4096^2 takes 296 us with
    // baselines up to 0.27 and 358 up to 0.45.
    constexpr int NZ = bfly_prunes(R0) ? (9 * R0 + 31) / 32 : R0 / 2;
    if constexpr (NZ < R0 / 2) {
        if (m.r1max < NZ * NB0) {
            transform(std::integral_constant<int, NZ>{});
            return;
        }
    }
    transform(std::integral_constant<int, R0 / 2>{});
}

template <int G, int KR>
__global__ __launch_bounds__(ColShape<G>::NX, ColShape<G>::waves) void k_stage1(
    const VisRec* __restrict__ sorted, const int* __restrict__ bstart, const SnapMeta* __restrict__ meta,
    const float2* __restrict__ tw, float2* __restrict__ kt, size_t stride)
{
    using Sh = ColShape<G>;
    __shared__ __align__(16) unsigned char smem[Sh::bytes];
    __shared__ float sc[Sh::NBLK], isc[Sh::NBLK];
    // Column-major over snapshots: the heavily populated low columns of
    // every snapshot are dispatched first, so none of them ends the launch.
    // On two axes: one of (g/2 + 1) S workgroups would pass the 2^32 threads
    // that an axis may hold from 43241 snapshots of 128^2 or 5455 of 1024^2 on.
    const int s = (int)blockIdx.x;
    const int c = (int)blockIdx.y;
    // The runs do not depend on the metadata: both loads are in flight
    // together.
    const int4 rg = column_ranges<G>(bstart + (size_t)s * boff_row(G), c);
    const SnapMeta m = meta[s];
    if (c > m.rmax) return;
    stage1_column<G, KR>(s, c, rg, sorted, m, tw, kt, stride, smem, sc, isc);
}

// ---------------------------------------------------------------- stage 2

// First K tile run of image row y0 of snapshot s.
template <int M>
__device__ __forceinline__ const float2* c2r_rows(const float2* __restrict__ kt, int s, int y0, int I)
{
    const float2* ks = kt + (size_t)s * ((size_t)I * (M + 1));
    return ks + (size_t)(y0 / kKTile) * (M + 1) * kKTile + (y0 % kKTile);
}

// Grid correction and output of two image rows from the transform's registers:
// real part the first row, imaginary part the second.  Element n of the
// transform is image column x = n (n < h) or n - g (n >= g - h), offset by h;
// with h = g/3 and the last radix a multiple of 3 the crop drops whole outputs
// of each butterfly.  |.| and 1/(c(|x|) c(|y|) norm^2) (FIPkernels.cu:256-287).
template <int G>
struct RowStore {
    static constexpr int I = 2 * G / 3, h = I / 2;
    static constexpr int R = FftPlan<G>::radix[FftPlan<G>::nstages - 1], NS = G / R, KEEP = R / 3;
    static_assert(R % 3 == 0 && 3 * h == G, "whole outputs are cropped");
    const float* __restrict__ corr;
    float* out;      // first row
    float cy0, cy1;
    float lmax;      // of this thread's butterfly
    float cv[2 * KEEP];

    __device__ __forceinline__ void prefetch(int j)
    {
        lmax = 0.0f;
        if (j >= NS) return;
#pragma unroll
        for (int k = 0; k < KEEP; ++k) {
            cv[k] = corr[NS * k + j];                                  // x = n
            cv[KEEP + k] = corr[(G - NS * (2 * KEEP + k)) - j];        // x = n - g
        }
    }
    __device__ __forceinline__ void operator()(int j, const float2* v)
    {
#pragma unroll
        for (int k = 0; k < 2 * KEEP; ++k) {
            const float2 z = v[k < KEEP ? k : k + KEEP];
            float* o = out + (k < KEEP ? h + NS * k : h + NS * (k + KEEP) - G) + j;
            const float a = fabsf(z.x) * (cv[k] * cy0), b = fabsf(z.y) * (cv[k] * cy1);
            // Non-temporal stores: 122-127 -> 108-109 us at 4096^2 for the row
            // pass, and the splat that reads these images next is not slower.
            __builtin_nontemporal_store(a, o);
            __builtin_nontemporal_store(b, o + I);
            lmax = fmaxf(lmax, fmaxf(a, b));
        }
    }
};

// Two image rows in one complex transform of length g: with Z[n] = K1[n] + i K2[n]
// over the whole Hermitian band (K[-n] = conj(K[n])), its real and imaginary
// parts are the two rows.  Each K entry of the pair is one 16-byte load, there
// is no split factor, the band (|n| <= cmax) leaves first-stage inputs out, and
// the crop leaves from the registers: one LDS pass in, two exchanges.  (A
// real transform per row as a complex one of half the length took its pairing
// factors, a full-length gather and two more LDS passes.)  K[0] and K[g/2] are
// real for exact data; their real parts are taken, so no row leaks into the
// other.
//
// Three images, before and after (rocprofv3): 96 -> 86 us at 4096^2 (339 MB, 3.9
// TB/s), 25 -> 24 at 2048^2.  Arithmetic and LDS turns of the waves (52 us of vector
// instructions) and the start of each workgroup on cold loads bound it now.
// Next rows' K loads held across the transform (a persistent loop) took 112
// registers instead of 70, with fewer waves and no gain.
//
// Workgroup: one row pair.  (Two pairs per workgroup: 3.7 -> 4.3 us at 128^2,
// 4.1 -> 4.3 at 256^2, within 6% either way from 512^2 to 2048^2, and the
// compiler contracts the two bodies differently, so the bits differ.)
template <int G>
__global__ __launch_bounds__(FftPlan<G>::nt, G >= 6144 ? 6 : 2) void k_stage2(
    const float2* __restrict__ kt, const SnapMeta* __restrict__ meta, unsigned* __restrict__ pmax,
    const float2* __restrict__ tw, const float* __restrict__ corr, float* __restrict__ pre)
{
    constexpr int M = G / 2, I = 2 * G / 3, h = I / 2, NT = FftPlan<G>::nt;
    constexpr int R0 = FftPlan<G>::radix[0], NB0 = G / R0;
    __shared__ float2 z[lds_len(G)];
    __shared__ unsigned shm[NT / 64];
    const int s = blockIdx.y, t = threadIdx.x;
    const int y0 = xcd_remap(blockIdx.x, gridDim.x) * 2;
    const int cmax = min(meta[s].rmax, M);
    const float2* k0 = c2r_rows<M>(kt, s, y0, I);
    RowStore<G> rows;
    rows.corr = corr;
    rows.out = pre + (size_t)s * I * I + (size_t)y0 * I;
    rows.cy0 = corr[y0 < h ? h - y0 : y0 - h];
    rows.cy1 = corr[y0 + 1 < h ? h - y0 - 1 : y0 + 1 - h];
    if (RowStore<G>::NS < NT) rows.lmax = 0.0f;   // threads without a last butterfly
    // NZ: first-stage inputs 0..NZ-1 and R0-NZ..R0-1, |n| <= NZ NB0.
    auto run = [&](auto NZ) {
        constexpr int nz = decltype(NZ)::value, L = nz * NB0, NIT = (L + NT - 1) / NT;
        auto pair = [&](int p) {
            return p <= cmax ? *reinterpret_cast<const float4*>(k0 + (size_t)p * kKTile)
                             : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        };
        float4 k[NIT];
#pragma unroll
        for (int u = 0; u < NIT; ++u)
            if (L % NT == 0 || t + u * NT < L) k[u] = pair(t + u * NT);
#pragma unroll
        for (int u = 0; u < NIT; ++u) {
            const int p = t + u * NT;
            if (L % NT == 0 || p < L) {
                if (p == 0) {
                    z[lds_pad(0)] = make_float2(k[u].x, k[u].z);
                    const float4 e = pair(L);   // g/2, or the band's first empty place
                    z[lds_pad(G - L)] = make_float2(e.x, e.z);
                } else {
                    z[lds_pad(p)] = make_float2(k[u].x - k[u].w, k[u].y + k[u].z);
                    z[lds_pad(G - p)] = make_float2(k[u].x + k[u].w, k[u].z - k[u].y);
                }
            }
        }
        __syncthreads();
        constexpr unsigned mask = band_mask<R0, nz, nz>();
        fft_inverse_io<G, true, false, mask>(
            z, tw, t, [&](int j, int r) { return lds_input<G, R0>(z, j, r); }, rows);
    };
    // The same band limit as the column pass: 9/32 of the grid on either side.
    constexpr int NZ = bfly_prunes(R0) ? (9 * R0 + 31) / 32 : R0 / 2;
    if (NZ < R0 / 2 && cmax < NZ * NB0)
        run(std::integral_constant<int, NZ>{});
    else
        run(std::integral_constant<int, R0 / 2>{});
    const unsigned bm = block_max_u<NT>(__float_as_uint(rows.lmax), shm);
    if (t == 0) atomicMax(max_slot(pmax, s, 0, (int)(blockIdx.x % kMaxSlots)), bm);
}

// Two image rows as in k_stage2, in two transforms of half the length: for
// 8192^2, where one of length 12288 would hold 101 KB of LDS, one workgroup per
// CU.  With X[x] = sum_n Z[n] e^{2 pi i n x/g}, M = g/2 and w = e^{2 pi i/g},
//   X[2m]     = sum_{n < M} (Z[n] + Z[n-M]) e^{2 pi i n m/M}
//   X[2m + 1] = sum_{n < M} (Z[n] - Z[n-M]) w^n e^{2 pi i n m/M}
// A thread takes the pairs (p, q = M - p): K[p] and K[q] give Z[+-p] and
// Z[+-q], all that elements p and q of both sums need (w^q = -conj(w^p)).  The
// second sum's inputs stay in registers through the first transform and its
// outputs through the second, so each K entry is read once, 16 bytes for both
// rows, and a row's columns 2m and 2m + 1 leave as one 8-byte store.
//
// Three images: 577 -> 467 us (1.46 GB, 3.1 TB/s) against one row per workgroup
// as a real transform, whose 8-byte loads each touched a 64-byte piece of the
// tiles.  119 registers, two workgroups per CU: the transforms' barriers are
// not always covered.
template <int G>
__global__ __launch_bounds__(FftPlan<G / 2>::nt, 4) void k_stage2_split(
    const float2* __restrict__ kt, const SnapMeta* __restrict__ meta, unsigned* __restrict__ pmax,
    const float2* __restrict__ tw, const float2* __restrict__ wpost, const float* __restrict__ corr,
    float* __restrict__ pre)
{
    constexpr int M = G / 2, I = 2 * G / 3, h = I / 2, NT = FftPlan<M>::nt;
    constexpr int R0 = FftPlan<M>::radix[0];
    constexpr int R = FftPlan<M>::radix[FftPlan<M>::nstages - 1], NS = M / R, KEEP = R / 3;
    constexpr int PB = (M / 2 + NT) / NT;   // pairs per thread: ceil((M/2 + 1)/NT)
    static_assert(R % 3 == 0 && 3 * h == G, "whole outputs are cropped");
    static_assert(NS == NT, "one last butterfly per thread");
    __shared__ float2 z[lds_len(M)];
    __shared__ unsigned shm[NT / 64];
    const int s = blockIdx.y, t = threadIdx.x;
    const int y0 = xcd_remap(blockIdx.x, gridDim.x) * 2;
    const int cmax = min(meta[s].rmax, M);
    const float2* k0 = c2r_rows<M>(kt, s, y0, I);
    float2 op[PB], oq[PB];   // the second sum's inputs p and q
    {
        float4 a[PB], b[PB];
        float2 wv[PB];
        auto load = [&](bool ok, int n) {
            return ok && n <= cmax ? *reinterpret_cast<const float4*>(k0 + (size_t)n * kKTile)
                                   : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        };
#pragma unroll
        for (int u = 0; u < PB; ++u) {
            const int p = t + u * NT;
            const bool ok = p <= M / 2;
            a[u] = load(ok, p);
            b[u] = load(ok, M - p);
            wv[u] = ok ? wpost[p] : make_float2(0.0f, 0.0f);
        }
#pragma unroll
        for (int u = 0; u < PB; ++u) {
            const int p = t + u * NT;
            if (p > M / 2) break;
            const float4 av = a[u], bv = b[u];
            if (p == 0) {
                // K[0] and K[g/2] are real
                z[lds_pad(0)] = make_float2(av.x + bv.x, av.z + bv.z);
                op[u] = make_float2(av.x - bv.x, av.z - bv.z);
                continue;
            }
            const float2 zp = make_float2(av.x - av.w, av.y + av.z), zmp = make_float2(av.x + av.w, av.z - av.y);
            const float2 zq = make_float2(bv.x - bv.w, bv.y + bv.z), zmq = make_float2(bv.x + bv.w, bv.z - bv.y);
            z[lds_pad(p)] = cadd(zp, zmq);
            op[u] = cmul(csub(zp, zmq), wv[u]);
            if (p != M - p) {
                z[lds_pad(M - p)] = cadd(zq, zmp);
                oq[u] = cmul(csub(zq, zmp), make_float2(-wv[u].x, wv[u].y));
            }
        }
    }
    __syncthreads();
    float2 even[2 * KEEP];
    auto in = [&](int j, int r) { return lds_input<M, R0>(z, j, r); };
    fft_inverse_io<M, true, false>(z, tw, t, in, [&](int, const float2* v) {
#pragma unroll
        for (int k = 0; k < 2 * KEEP; ++k) even[k] = v[k < KEEP ? k : k + KEEP];
    });
    __syncthreads();   // the last stage has read z
#pragma unroll
    for (int u = 0; u < PB; ++u) {
        const int p = t + u * NT;
        if (p > M / 2) break;
        z[lds_pad(p)] = op[u];
        if (p != 0 && p != M - p) z[lds_pad(M - p)] = oq[u];
    }
    __syncthreads();
    const float cy0 = corr[y0 < h ? h - y0 : y0 - h], cy1 = corr[y0 + 1 < h ? h - y0 - 1 : y0 + 1 - h];
    float* const row = pre + (size_t)s * I * I + (size_t)y0 * I;
    float lmax = 0.0f;
    fft_inverse_io<M, true, false>(z, tw, t, in, [&](int j, const float2* v) {
#pragma unroll
        for (int k = 0; k < 2 * KEEP; ++k) {
            const int r = k < KEEP ? k : k + KEEP;
            const int x = 2 * (j + NS * r) - (k < KEEP ? 0 : G);
            const float c0 = corr[x < 0 ? -x : x], c1 = corr[x < 0 ? -x - 1 : x + 1];
            typedef float fip_f2 __attribute__((ext_vector_type(2)));
            const fip_f2 v0 = {fabsf(even[k].x) * (c0 * cy0), fabsf(v[r].x) * (c1 * cy0)};
            const fip_f2 v1 = {fabsf(even[k].y) * (c0 * cy1), fabsf(v[r].y) * (c1 * cy1)};
            __builtin_nontemporal_store(v0, reinterpret_cast<fip_f2*>(row + (x + h)));
            __builtin_nontemporal_store(v1, reinterpret_cast<fip_f2*>(row + I + (x + h)));
            lmax = fmaxf(fmaxf(lmax, fmaxf(v0.x, v0.y)), fmaxf(v1.x, v1.y));
        }
    });
    const unsigned bm = block_max_u<NT>(__float_as_uint(lmax), shm);
    if (t == 0) atomicMax(max_slot(pmax, s, 0, (int)(blockIdx.x % kMaxSlots)), bm);
}

// ----------------------------------------------------------------- splat

__device__ __forceinline__ void sin_shift(const SnapGeom& g, double q1, double q2, double& o1, double& o2)
{
    o1 = q1;
    o2 = q2;
    if (!g.sin_on) return;
    // l = -cell (P1 - c0), m = cell (P2 - c0), c0 = I/2 + 1 (FIPkernels.cu:315-316)
    const float l = (float)(-g.delta * (q1 - 1.0));
    const float mm = (float)(g.delta * (q2 - 1.0));
    const float r2 = l * l + mm * mm;
    if (g.series) {
        // every source of the image has r^2 <= 0.01 (checked in snap_geometry)
        const float np = r2 * fmaf(r2, fmaf(r2, fmaf(r2, 0.0390625f, 0.0625f), 0.125f), 0.5f);
        o1 = q1 + g.sx * (double)np;
        o2 = q2 + g.sy * (double)np;
    } else if (r2 <= 1.0f) {
        // 1 - sqrt(1 - r^2) = r^2 / (1 + sqrt(1 - r^2)); hardware sqrt/rcp (1 ulp)
        const float np = r2 * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_sqrtf(1.0f - r2));
        o1 = q1 + g.sx * (double)np;
        o2 = q2 + g.sy * (double)np;
    }
}

// a * b + c for a, b < 2^24 in one full-rate instruction (the compiler
// otherwise forms a quarter-rate 32-bit multiply).
__device__ __forceinline__ unsigned mad_u24(unsigned a, unsigned b, unsigned c)
{
    unsigned r;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// a * b + c for |a|, |b| < 2^23 (signed 24-bit) in one full-rate instruction;
// b is uniform (a scalar register).
__device__ __forceinline__ int mad_i24(int a, int b, int c)
{
    int r;
    asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
}

// Exact integer accumulation: contributions (non-negative) are scaled by a
// power of two, rounded half up to integers and summed as int32; the scale
// keeps every pixel sum below 2^29 (plus half a unit per contribution), so
// each sum is exact and independent of the order of the LDS atomics.
__device__ __forceinline__ void acc_exact(int* a, float x)
{
    atomicAdd(a, cvt_round_half_up_i32(x));
}

// Non-temporal 16-byte load for the trigger, which reads each image byte
// once.  Measured on the one-window trigger: 157 -> 128 us at 8192^2 (three
// images of 268 MB), unchanged at 4096^2; same bits.
typedef float fip_f4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 load_stream(const float* p)
{
    const fip_f4 v = __builtin_nontemporal_load(reinterpret_cast<const fip_f4*>(p));
    return make_float4(v.x, v.y, v.z, v.w);
}

// Trigger terms of one pixel (FIPkernels.cu:499-552): dd = ||a - b| - |b - c||,
// its sum and maximum, and the sum of the guarded ratio min(dd / b', 1) with
// b' = b, or 1e-6 where b <= 0 (FIPkernels.cu:811).  Every trigger form adds
// a lane's pixels in the same order through this function, so their sums
// agree bit for bit.
__device__ __forceinline__ void tlisi_px(float a, float b, float c, float& sum, float& mx, float& sr)
{
    const float dd = fabsf(fabsf(a - b) - fabsf(b - c));
    const float b2 = (b <= 0.0f) ? 1e-6f : b;
    sum += dd;
    mx = fmaxf(mx, dd);
    const float ratio = dd / b2;
    sr += (ratio < 1.0f) ? ratio : 1.0f;
}

// tLISI of a T x T tile from its reduced terms and the window's maximum m3
// (FIPkernels.cu:550).
__device__ __forceinline__ float tlisi_value(float sum, float mx, float sr, float m3, int T)
{
    const float Tf = (float)T;
    return 1.0f - (sum / Tf / Tf) * mx * (sr / Tf / Tf) / m3 / m3;
}

// Per target tile: bounding box and per-row ranges of the source pixels whose
// bilinear footprint can reach the tile, then the forward splat
// (finalinterp, FIPkernels.cu:378-413) accumulated in an LDS tile with a
// one-pixel apron.  The candidate sources of a batch of rows are numbered
// row by row; lane work is a contiguous range of that numbering, so every
// lane of every wave has a source whatever the rotation of the map.  A
// lane finds its row from a table of the rows in which each run of 64
// numbers starts (usually no further step) and keeps four independent
// loads and position chains in flight; at most 64 VGPRs keep eight waves
// per SIMD resident.  Snapshot s0 + blockIdx.y.
//
// TRIG: the last snapshot of a three-snapshot window with the trigger fused
// in.  Its image is stored only if store_img; each wave takes one 32 x 32
// trigger tile of the 64 x 64 target tile, reads the window's first two
// images (img_a, img_b, written by an earlier launch) and this tile's values
// from LDS, and stores the tile's reduced terms (sum, max, ratio sum) to part;
// the tLISI follows once every image maximum is known (k_trigger_finish).
template <int TS, bool TRIG>
__global__ __launch_bounds__(256, 8) void k_splat(const float* __restrict__ pre, const SnapMeta* __restrict__ meta,
                                               const SnapGeom* __restrict__ geom, unsigned* __restrict__ pmax,
                                               float* __restrict__ img, int I, int s0,
                                               const float* __restrict__ img_a, const float* __restrict__ img_b,
                                               float* __restrict__ part, int store_img)
{
    constexpr int NT = 256;
    constexpr int NW = NT / 64;           // waves
    constexpr int ROW_CAP = 2 * TS + 32;   // source rows handled per pass
    constexpr int A = TS + 2;             // apron: targets -1 .. TS
    constexpr int GN = 8;                 // consecutive sources of a row per lane
    constexpr int CHK = 512;              // runs of 64 numbered groups per window
    static_assert(GN % 4 == 0 && (GN & (GN - 1)) == 0, "groups of 16-byte loads");
    static_assert((A * A) % 4 == 0, "16-byte clears");
    static_assert(NW == 4 && ROW_CAP < NT, "one row per thread");
    __shared__ __align__(16) int acc[A * A];
    __shared__ int rlo[ROW_CAP], rofs[ROW_CAP + 1];
    __shared__ unsigned char crow[CHK];   // row in which each run of 64 starts
    __shared__ double qb[6];
    __shared__ int bb[4];
    __shared__ __align__(16) int wtot[NW];
    __shared__ unsigned shm[NT / 64];
    __shared__ float sscale[2];
    const int s = s0 + (int)blockIdx.y;
    const int ntx = I / TS;
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int R0 = (tile / ntx) * TS, C0 = (tile % ntx) * TS;
    const SnapGeom& g = geom[s];
    const int h = I / 2;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    if (tid == 0) {
        int i0 = 0, i1 = I - 1, j0 = 0, j1 = I - 1;
        // q-space (affine position - h) box that can reach the open target box
        // (C0-1, C0+TS) x (R0-1, R0+TS): the target box shifted by the SIN
        // shift at the tile centre, widened by its variation over the tile.
        double ql1 = -1e300, qh1 = 1e300, ql2 = -1e300, qh2 = 1e300;
        if (g.curv >= 0.0) {
            const double t1 = (double)C0 + 0.5 * (TS - 1) - h, t2 = (double)R0 + 0.5 * (TS - 1) - h;
            double q1 = t1, q2 = t2;
            // At most four fixed-point steps; the residual below bounds what is
            // left, so stopping once a step moves less than 1e-4 px keeps the
            // box conservative.
            for (int it = 0; it < 4; ++it) {
                double o1, o2;
                sin_shift(g, q1, q2, o1, o2);
                const double n1 = t1 - (o1 - q1), n2 = t2 - (o2 - q2);
                const bool done = fabs(n1 - q1) + fabs(n2 - q2) < 1e-4;
                q1 = n1;
                q2 = n2;
                if (done) break;
            }
            double o1, o2;
            sin_shift(g, q1, q2, o1, o2);
            const double d1 = o1 - q1, d2 = o2 - q2;
            // Any q with q + d(q) in the box lies within (halfdiag + residual)/(1 - kappa)
            // of (q1, q2), so |d(q) - d| <= kappa times that.
            const double res = fabs(o1 - t1) + fabs(o2 - t2);
            const double halfdiag = 0.7071067811865476 * (TS + 1);
            const double dv = g.kratio * (halfdiag + res) + 0.02;
            ql1 = (double)(C0 - 1) - h - d1 - dv;
            qh1 = (double)(C0 + TS) - h - d1 + dv;
            ql2 = (double)(R0 - 1) - h - d2 - dv;
            qh2 = (double)(R0 + TS) - h - d2 + dv;
            // Extent of the inverse map over the box: each term's own extremes.
            auto extent = [&](double ca, double cb, double& lo, double& hi) {
                const double a0 = ca * ql1, a1 = ca * qh1, b0 = cb * ql2, b1 = cb * qh2;
                lo = fmin(a0, a1) + fmin(b0, b1) + h;
                hi = fmax(a0, a1) + fmax(b0, b1) + h;
                // clamp before converting (degenerate V can give huge values)
                lo = fmin(fmax(lo, -4.0), (double)I + 4.0);
                hi = fmin(fmax(hi, -4.0), (double)I + 4.0);
            };
            double mini, maxi, minj, maxj;
            extent(g.i00, g.i01, mini, maxi);
            extent(g.i10, g.i11, minj, maxj);
            i0 = max(0, (int)floor(mini) - 1);
            i1 = min(I - 1, (int)ceil(maxi) + 1);
            j0 = max(0, (int)floor(minj) - 1);
            j1 = min(I - 1, (int)ceil(maxj) + 1);
        }
        qb[0] = ql1;
        qb[1] = qh1;
        qb[2] = ql2;
        qb[3] = qh2;
        qb[4] = g.im00;
        qb[5] = g.im10;
        bb[0] = i0;
        bb[1] = i1;
        bb[2] = j0;
        bb[3] = j1;
    }
    {
        int4* a4 = reinterpret_cast<int4*>(acc);
        for (int q = tid; q < A * A / 4; q += NT) a4[q] = make_int4(0, 0, 0, 0);
    }
    if (wid == 1) {
        // While thread 0 computes the box: the max of the corrected image
        // from its slots (one per lane), and the scale.  A pixel sums at most
        // ccap contributions of at most max(pre)/N each (1/N of
        // FIPkernels.cu:391); 2^k * ccap * max(pre)/N < 2^29.
        const float maxp = __uint_as_float(wave_max_u(*max_slot(pmax, s, 0, lane)));
        const float nf = (float)meta[s].norm_n;
        int e = 0;
        frexpf(fmaxf((float)g.ccap * (maxp / nf), 1e-30f), &e);
        const int ks = min(29 - e, 120);
        if (lane == 0) {
            sscale[0] = ldexpf(1.0f, ks) / nf;
            sscale[1] = ldexpf(1.0f, -ks);
        }
    }
    __syncthreads();
    const int i0 = bb[0], i1 = bb[1], j0 = bb[2], j1 = bb[3];
    // Accepted target offsets of a footprint's top-left corner: the apron
    // -1..TS-1 intersected with |LL| < h - 1, i.e. floor(LL) in [1-h, h-2]
    // (floor(LL) >= 2-h when LL is an integer).
    const int cxlo = max(-1, 1 - C0), cxn = min(TS - 1, I - 2 - C0) - cxlo;
    const int rylo = max(-1, 1 - R0), ryn = min(TS - 1, I - 2 - R0) - rylo;
    const bool cedge = 1 - C0 >= -1, redge = 1 - R0 >= -1;   // tile on the left / top image edge
    // Without a curvature bound positions are not bounded a priori.
    const bool unbounded = g.curv < 0.0;
    const int H = j1 - j0 + 1;
    const float vscale = sscale[0], iscale = sscale[1];
    const float* ps = pre + (size_t)s * I * I;
    for (int rb = 0; rb < H; rb += ROW_CAP) {
        const int nrow = min(ROW_CAP, H - rb);
        // Per source row, one thread: the i range whose affine position lies
        // in the q box, in groups of GN pixels aligned to i % GN == 0, and
        // their running count over the rows (DPP within a wave, the waves'
        // totals through LDS).
        int first = 0, cnt = 0;
        if (tid < nrow) {
            const double b = (double)(j0 + rb + tid - h);
            double alo = -1e300, ahi = 1e300;
            const double mA[2] = {g.m00, g.m10}, mB[2] = {g.m01, g.m11}, iA[2] = {qb[4], qb[5]};
            // The q box is read from LDS here rather than held in registers
            // across the source loop (eight VGPRs; holding them spilled).
            const double lo[2] = {qb[0], qb[2]}, hi[2] = {qb[1], qb[3]};
            for (int k = 0; k < 2; ++k) {
                const double cst = mB[k] * b;
                if (fabs(mA[k]) > 1e-12) {
                    // The range is widened by one pixel below, so a rounded
                    // reciprocal is as good as a division here.
                    const double x = (lo[k] - cst) * iA[k], y = (hi[k] - cst) * iA[k];
                    alo = fmax(alo, fmin(x, y));
                    ahi = fmin(ahi, fmax(x, y));
                } else if (cst < lo[k] || cst > hi[k]) {
                    alo = 1e300;
                    ahi = -1e300;
                }
            }
            alo = fmax(alo, (double)(i0 - h - 2));
            ahi = fmin(ahi, (double)(i1 - h + 2));
            if (alo <= ahi) {
                const int ia = max(i0, (int)floor(alo + h) - 1);
                const int n = max(0, min(i1, (int)ceil(ahi + h) + 1) - ia + 1);
                first = ia / GN;
                cnt = n > 0 ? ((ia + n - 1) / GN) - first + 1 : 0;
            }
        }
        const int incl = wave_scan_i(cnt);
        if (lane == 63) wtot[wid] = incl;
        __syncthreads();
        int ofs = incl - cnt, total = 0;
        {
            const int4 w = *reinterpret_cast<const int4*>(wtot);
            ofs += (wid > 0 ? w.x : 0) + (wid > 1 ? w.y : 0) + (wid > 2 ? w.z : 0);
            total = __builtin_amdgcn_readfirstlane(w.x + w.y + w.z + w.w);
        }
        if (tid < nrow) {
            rlo[tid] = first;
            rofs[tid] = ofs;
        }
        if (tid == nrow) rofs[nrow] = total;
        for (int f0 = 0; f0 < total; f0 += CHK * 64) {
            const int nf = min(CHK * 64, total - f0);
            // Row of the first number of every run of 64 in [f0, f0 + nf).
            if (tid < nrow) {
                const int a = max(ofs, f0), b = min(ofs + cnt, f0 + nf);
                for (int k = (a - f0 + 63) >> 6; (k << 6) < b - f0; ++k) crow[k] = (unsigned char)tid;
            }
            __syncthreads();
            // The source loop, specialised on the tile: EDGE for tiles on the
            // left or top image edge (an integer position on the bound is
            // outside there), UNB for maps without a curvature bound
            // (positions checked for size).  Interior tiles of bounded maps,
            // nearly all of them, take neither check.
            auto sources = [&](auto EDGE, auto UNB, auto SER) {
                constexpr bool edge = decltype(EDGE)::value, unb = decltype(UNB)::value;
                // SIN shift: 1 by its series, 0 by its closed form (a map
                // without one has sx = sy = 0, which adds exact zeros), -1 as
                // the geometry's flags say
                constexpr int ser = decltype(SER)::value;
                for (int base = 0; base < nf; base += NT) {
                    const int fl = base + tid;
                    if (fl >= nf) break;
                    const int f = f0 + fl;
                    int r = crow[fl >> 6];
                    while (rofs[r + 1] <= f) ++r;
                    const int gi = rlo[r] + (f - rofs[r]);
                    const int jj = j0 + rb + r;
                    // Aligned 16-byte loads (I % GN == 0, so a group never
                    // crosses the end of a row).
                    float pv[GN];
                    const float4* src = reinterpret_cast<const float4*>(ps + (size_t)jj * I + GN * gi);
#pragma unroll
                    for (int u = 0; u < GN / 4; ++u) {
                        const float4 q = src[u];
                        pv[4 * u] = q.x;
                        pv[4 * u + 1] = q.y;
                        pv[4 * u + 2] = q.z;
                        pv[4 * u + 3] = q.w;
                    }
                    // Group origin in FP64: the affine position of its first
                    // pixel (clamped: positions beyond 1e6 px are rejected
                    // below), split into an integer part O and a fraction.  The
                    // pixels are placed in FP32 relative to O (local
                    // coordinates stay within a few pixels, ~1e-7 px), and only
                    // integer parts are recombined.
                    const double a0 = (double)(GN * gi - h), b = (double)(jj - h);
                    double q1d = fma(g.m00, a0, g.m01 * b), q2d = fma(g.m10, a0, g.m11 * b);
                    if constexpr (unb) {
                        // bounded maps keep positions within the image's reach
                        q1d = fmin(fmax(q1d, -1e6), 1e6);
                        q2d = fmin(fmax(q2d, -1e6), 1e6);
                    }
                    const double O1 = floor(q1d), O2 = floor(q2d);
                    const float r1 = (float)(q1d - O1), r2 = (float)(q2d - O2);
                    // target offsets of the origin in the tile, relative to the
                    // accepted ranges' starts, and the LDS byte address of the
                    // origin's apron cell
                    const int c1 = (int)O1 + h - C0, c2 = (int)O2 + h - R0;
                    const int e1 = c1 - cxlo, e2 = c2 - rylo;
                    unsigned gb = 4u * (unsigned)(__mul24(c2 + 1, A) + c1 + 1);
                    asm volatile("" : "+v"(gb));   // kept whole, so gb + 4 f1 is one instruction
                    // SIN direction cosines along the group: l = -cell (P1 - c0),
                    // m = cell (P2 - c0), c0 = I/2 + 1 (FIPkernels.cu:315-316),
                    // rounded once from FP64.
                    const float l0 = (float)fma(-g.delta, q1d, g.delta), dl = g.fdl;
                    const float n0 = (float)fma(g.delta, q2d, -g.delta), dn = g.fdn;
                    // Series form: source k of the group lands at
                    // (Q1 + B1 k + C1 k^2, Q2 + B2 k + C2 k^2) relative to the
                    // origin, the affine step plus the quadratic Taylor model in
                    // k of the SIN shift (sx, sy) n'(k) (its remainder is
                    // bounded in snap_geometry).  With r^2(k) = R0 + R1 k + R2 k^2 and
                    // the series f(x) = x/2 + x^2/8 + x^3/16 + 5x^4/128,
                    // n'(k) ~ f(R0) + f'(R0) R1 k + (f'(R0) R2 + f''(R0) R1^2 / 2) k^2.
                    float Q1 = r1, B1 = g.fm00, C1 = 0.0f, Q2 = r2, B2 = g.fm10, C2 = 0.0f;
                    if constexpr (ser == 1) {
                        const float R0 = fmaf(l0, l0, n0 * n0);
                        const float R1 = fmaf(l0, 2.0f * dl, n0 * (2.0f * dn));
                        const float R2 = fmaf(dl, dl, dn * dn);
                        const float f0 = R0 * fmaf(R0, fmaf(R0, fmaf(R0, 0.0390625f, 0.0625f), 0.125f), 0.5f);
                        const float f1 = fmaf(R0, fmaf(R0, fmaf(R0, 0.15625f, 0.1875f), 0.25f), 0.5f);
                        const float f2h = fmaf(R0, fmaf(R0, 0.234375f, 0.1875f), 0.125f);
                        const float b = f1 * R1, c = fmaf(f1, R2, f2h * R1 * R1);
                        Q1 = fmaf(g.fsx, f0, r1);
                        Q2 = fmaf(g.fsy, f0, r2);
                        B1 = fmaf(g.fsx, b, g.fm00);
                        B2 = fmaf(g.fsy, b, g.fm10);
                        C1 = g.fsx * c;
                        C2 = g.fsy * c;
                    }
#pragma unroll
                    for (int k = 0; k < GN; ++k) {
                        float o1, o2;
                        if constexpr (ser == 1) {
                            o1 = k == 0 ? Q1 : fmaf((float)(k * k), C1, fmaf((float)k, B1, Q1));
                            o2 = k == 0 ? Q2 : fmaf((float)(k * k), C2, fmaf((float)k, B2, Q2));
                        } else {
                            o1 = fmaf((float)k, g.fm00, r1);
                            o2 = fmaf((float)k, g.fm10, r2);
                            if (ser == 0 || g.sin_on) {
                                const float l = fmaf((float)k, dl, l0), mm = fmaf((float)k, dn, n0);
                                const float rr = l * l + mm * mm;
                                float np = 0.0f;
                                if (ser < 0 && g.series) {
                                    // every source of the image has r^2 <= 0.01 (checked in snap_geometry)
                                    np = rr * fmaf(rr, fmaf(rr, fmaf(rr, 0.0390625f, 0.0625f), 0.125f), 0.5f);
                                } else if (rr <= 1.0f) {
                                    // 1 - sqrt(1 - r^2) = r^2 / (1 + sqrt(1 - r^2)); hardware sqrt/rcp
                                    np = rr * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_sqrtf(1.0f - rr));
                                }
                                o1 = fmaf(g.fsx, np, o1);
                                o2 = fmaf(g.fsy, np, o2);
                            }
                        }
                        bool fin = true;
                        if constexpr (unb) {
                            // finite and small enough for the integer recombination
                            fin = fabsf(o1) < 1048576.0f && fabsf(o2) < 1048576.0f;
                            o1 = fin ? o1 : 0.0f;
                            o2 = fin ? o2 : 0.0f;
                        }
                        // floor as an integer and the fraction o - floor(o) in
                        // [0, 1): the bilinear weights of the two axes
                        const int f1 = cvt_floor_i32(o1), f2 = cvt_floor_i32(o2);
                        const float wl1 = __builtin_amdgcn_fractf(o1), wm1 = __builtin_amdgcn_fractf(o2);
                        // Tile apron and |LL|, |MM| < h - 1 (FIPkernels.cu:389) as
                        // one unsigned range per axis; on the left / top image
                        // edge an integer position on the bound is outside.
                        const int u1 = f1 + e1, u2 = f2 + e2;
                        bool ok = (unsigned)u1 <= (unsigned)cxn && (unsigned)u2 <= (unsigned)ryn;
                        if constexpr (unb) ok = ok && fin;
                        if constexpr (edge)
                            ok = ok && !(cedge && u1 == 0 && wl1 == 0.0f) && !(redge && u2 == 0 && wm1 == 0.0f);
                        if (ok) {
                            // FIPkernels.cu:395-410: (fM,fL), (cM,fL), (fM,cL), (cM,cL)
                            // with weights (1-a)(1-b), (1-a)b, a(1-b), ab; each
                            // product is split off its row by one subtraction.  A
                            // zero weight on an integer position adds an exact zero.
                            const float vs = pv[k] * vscale;
                            const float t1 = wl1 * vs, t0 = vs - t1;
                            const float p01 = t0 * wm1, p11 = t1 * wm1;
                            const float p00 = t0 - p01, p10 = t1 - p11;
                            int* p0 = reinterpret_cast<int*>(reinterpret_cast<char*>(acc) +
                                                             (unsigned)mad_i24(f2, 4 * A, (int)gb + 4 * f1));
                            acc_exact(p0, p00);
                            acc_exact(p0 + A, p01);
                            acc_exact(p0 + 1, p10);
                            acc_exact(p0 + A + 1, p11);
                        }
                    }
                }
            };
            // Bounded maps take the SIN form as a compile-time choice: 2-5%
            // faster than the per-source test of the flags.
            using Series = std::integral_constant<int, 1>;
            using Closed = std::integral_constant<int, 0>;
            if (unbounded) {
                sources(std::true_type{}, std::true_type{}, std::integral_constant<int, -1>{});
            } else if (cedge || redge) {
                if (g.series)
                    sources(std::true_type{}, std::false_type{}, Series{});
                else
                    sources(std::true_type{}, std::false_type{}, Closed{});
            } else {
                if (g.series)
                    sources(std::false_type{}, std::false_type{}, Series{});
                else
                    sources(std::false_type{}, std::false_type{}, Closed{});
            }
            __syncthreads();   // crow is rewritten by the next window
        }
        if (rb + ROW_CAP < H) __syncthreads();   // rlo/rofs/wtot are rewritten by the next row batch
    }
    float* out = img + (size_t)s * I * I;
    int lmax = 0;   // the scale is positive: the largest sum is the largest value
    // Four consecutive pixels per thread per pass, one 16-byte store; each
    // pass covers NT / (TS / 4) rows, and the pointers step by that.
    {
        constexpr int RSTEP = NT / (TS / 4);
        static_assert((TS * TS / 4) % NT == 0, "whole passes");
        const int rr = tid / (TS / 4), cc = 4 * (tid % (TS / 4));
        const int* a = acc + (rr + 1) * A + cc + 1;
        float* o = out + (size_t)(R0 + rr) * I + C0 + cc;
#pragma unroll
        for (int q = 0; q < TS * TS / 4 / NT; ++q) {
            const float4 v = make_float4((float)a[0] * iscale, (float)a[1] * iscale, (float)a[2] * iscale,
                                         (float)a[3] * iscale);
            if (!TRIG || store_img) *reinterpret_cast<float4*>(o) = v;
            lmax = max(max(lmax, max(a[0], a[1])), max(a[2], a[3]));
            a += RSTEP * A;
            o += (size_t)RSTEP * I;
        }
    }
    const unsigned bmx = block_max_u<NT>(__float_as_uint((float)lmax * iscale), shm);
    if (tid == 0) atomicMax(max_slot(pmax, s, 1, (int)(blockIdx.x % kMaxSlots)), bmx);
    if constexpr (TRIG) {
        // The trigger tile of this wave; lanes take the pixels, and add them
        // in the order, of k_trigger (16-byte groups lane + 64 u), so the
        // reduced terms are the same bits as k_trigger's.
        static_assert(TS == 64, "four 32 x 32 trigger tiles per workgroup, one per wave");
        constexpr int T = 32;
        const int tr = R0 + T * (wid >> 1), tc = C0 + T * (wid & 1);
        float sum = 0.0f, mx = 0.0f, sr = 0.0f;
        float4 av[4], bv[4], cv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int p = lane + 64 * u, row = p / (T / 4), col = 4 * (p % (T / 4));
            const size_t q = (size_t)(tr + row) * I + (size_t)(tc + col);
            av[u] = load_stream(img_a + q);
            bv[u] = load_stream(img_b + q);
            // the values this launch would have stored
            const int* ac = acc + (tr - R0 + row + 1) * A + (tc - C0 + col + 1);
            cv[u] = make_float4((float)ac[0] * iscale, (float)ac[1] * iscale, (float)ac[2] * iscale,
                                (float)ac[3] * iscale);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            tlisi_px(av[u].x, bv[u].x, cv[u].x, sum, mx, sr);
            tlisi_px(av[u].y, bv[u].y, cv[u].y, sum, mx, sr);
            tlisi_px(av[u].z, bv[u].z, cv[u].z, sum, mx, sr);
            tlisi_px(av[u].w, bv[u].w, cv[u].w, sum, mx, sr);
        }
        sum = wave_sum_f(sum);
        mx = wave_max_f(mx);
        sr = wave_sum_f(sr);
        if (lane == 0) {
            float* pp = part + 3 * ((size_t)(tr / T) * (I / T) + (size_t)(tc / T));
            pp[0] = sum;
            pp[1] = mx;
            pp[2] = sr;
        }
    }
}

// tLISI of one window from the fused splat's reduced terms: each wave reduces
// the window's three image maxima from their spread slots (as k_trigger does),
// then each thread finishes one tile.
__global__ __launch_bounds__(256) void k_trigger_finish(const float* __restrict__ part, SnapMeta* __restrict__ meta,
                                                        unsigned* __restrict__ pmax, int s1, int s2, int s3, int I,
                                                        int T, float* __restrict__ out)
{
    const int lane = threadIdx.x & 63;
    const unsigned m1b = wave_max_u(*max_slot(pmax, s1, 1, lane)), m2b = wave_max_u(*max_slot(pmax, s2, 1, lane)),
                   m3b = wave_max_u(*max_slot(pmax, s3, 1, lane));
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        // the reduced maxima for host readers
        meta[s1].maxd_bits = m1b;
        meta[s2].maxd_bits = m2b;
        meta[s3].maxd_bits = m3b;
    }
    const int un = I / T;
    const int tile = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (tile >= un * un) return;
    const float* pp = part + 3 * (size_t)tile;
    const float m3 = fmaxf(__uint_as_float(m1b), fmaxf(__uint_as_float(m2b), __uint_as_float(m3b)));
    out[tile] = tlisi_value(pp[0], pp[1], pp[2], m3, T);
}

// --------------------------------------------------------------- trigger

// One wave per tile (four tiles per workgroup): per-lane partial sums over
// 16-byte loads, then wave reductions only (FIPkernels.cu:499-552).  A tile
// whose edge is no multiple of four pixels takes 4-byte loads, of eight turns
// together where a lane has more than two pixels: at tile 50 (40 pixels a lane)
// 20 -> 9 us at 1024^2, 19 -> 12 at 2048^2 and 43 -> 40 at 4096^2 (201 MB, 5
// TB/s); with one or two, the set-up would cost 2 to 5% (tile 3 to 9).
enum TriggerMode { kTrigWide, kTrigDeep, kTrigSmall };
template <TriggerMode MODE>
__global__ __launch_bounds__(256) void k_trigger(const float* __restrict__ img, SnapMeta* __restrict__ meta,
                                                 unsigned* __restrict__ pmax, const int* __restrict__ win, int I,
                                                 int T, TriggerOut out)
{
    const int w = blockIdx.y;
    const int un = I / T;
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile >= un * un) return;   // whole wave
    const int ti = tile / un, tj = tile % un;
    const int s1 = win[3 * w], s2 = win[3 * w + 1], s3 = win[3 * w + 2];
    // Image maxima from the spread slots (one slot per lane).
    const unsigned q1 = *max_slot(pmax, s1, 1, lane), q2 = *max_slot(pmax, s2, 1, lane),
                   q3 = *max_slot(pmax, s3, 1, lane);
    const float* d1 = img + (size_t)s1 * I * I;
    const float* d2 = img + (size_t)s2 * I * I;
    const float* d3 = img + (size_t)s3 * I * I;
    float sum = 0.0f, mx = 0.0f, sr = 0.0f;
    auto px = [&](float a, float b, float c) { tlisi_px(a, b, c, sum, mx, sr); };
    if constexpr (MODE == kTrigWide) {
        // 16-byte loads: rows of a tile start at multiples of 4 floats; the
        // loads of four passes are issued together.
        const int T4 = T >> 2, n4 = T * T4;
        for (int p0 = lane; p0 < n4; p0 += 4 * 64) {
            float4 a[4], b[4], c[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int p = p0 + u * 64;
                if (p < n4) {
                    const size_t q = (size_t)(ti * T + p / T4) * I + (size_t)(tj * T + 4 * (p % T4));
                    a[u] = load_stream(d1 + q);
                    b[u] = load_stream(d2 + q);
                    c[u] = load_stream(d3 + q);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (p0 + u * 64 < n4) {
                    px(a[u].x, b[u].x, c[u].x);
                    px(a[u].y, b[u].y, c[u].y);
                    px(a[u].z, b[u].z, c[u].z);
                    px(a[u].w, b[u].w, c[u].w);
                }
            }
        }
    } else if constexpr (MODE == kTrigDeep) {
        // eight turns' loads together, the places stepped instead of divided
        constexpr int U = 8;
        const int drow = 64 / T, dcol = 64 % T;
        int row = lane / T, col = lane % T;
        for (int p0 = lane; p0 < T * T; p0 += U * 64) {
            float a[U], b[U], c[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (p0 + u * 64 < T * T) {
                    const size_t q = (size_t)(ti * T + row) * I + (size_t)(tj * T + col);
                    a[u] = d1[q];
                    b[u] = d2[q];
                    c[u] = d3[q];
                }
                row += drow;
                col += dcol;
                if (col >= T) {
                    col -= T;
                    ++row;
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (p0 + u * 64 < T * T) px(a[u], b[u], c[u]);
        }
    } else {
        for (int p = lane; p < T * T; p += 64) {
            const size_t q = (size_t)(ti * T + p / T) * I + (size_t)(tj * T + p % T);
            px(d1[q], d2[q], d3[q]);
        }
    }
    sum = wave_sum_f(sum);
    mx = wave_max_f(mx);
    sr = wave_sum_f(sr);
    const unsigned m1b = wave_max_u(q1), m2b = wave_max_u(q2), m3b = wave_max_u(q3);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        // the reduced maxima for host readers (every window writes the same values)
        meta[s1].maxd_bits = m1b;
        meta[s2].maxd_bits = m2b;
        meta[s3].maxd_bits = m3b;
    }
    if (lane == 0) {
        const float m3 = fmaxf(__uint_as_float(m1b), fmaxf(__uint_as_float(m2b), __uint_as_float(m3b)));
        out.w[w][tile] = tlisi_value(sum, mx, sr, m3, T);
    }
}

// Consecutive windows (s0+w, s0+w+1, s0+w+2), w < nwin, of a batch: one wave
// per tile handles up to kRunWin consecutive windows, so each image is read
// once per kRunWin windows instead of three times per window.
constexpr int kRunWin = 8;

__global__ __launch_bounds__(256) void k_trigger_run(const float* __restrict__ img, SnapMeta* __restrict__ meta,
                                                     unsigned* __restrict__ pmax, int s0, int nwin, int I, int T,
                                                     float* __restrict__ out)
{
    constexpr int K = kRunWin, NI = kRunWin + 2;
    const int un = I / T;
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile >= un * un) return;   // whole wave
    const int w0 = blockIdx.y * K, nk = min(K, nwin - w0), ni = nk + 2;
    const int i0 = s0 + w0;
    const int ti = tile / un, tj = tile % un;
    // Image maxima from the spread slots (one slot per lane).
    unsigned md[NI];
#pragma unroll
    for (int j = 0; j < NI; ++j) md[j] = wave_max_u(j < ni ? *max_slot(pmax, i0 + j, 1, lane) : 0u);
    float sum[K], mx[K], sr[K];
#pragma unroll
    for (int k = 0; k < K; ++k) sum[k] = mx[k] = sr[k] = 0.0f;
    auto px = [&](int k, float a, float b, float c) { tlisi_px(a, b, c, sum[k], mx[k], sr[k]); };
    const size_t plane = (size_t)I * I;
    const float* base = img + (size_t)i0 * plane;
    if ((T & 3) == 0) {
        const int T4 = T >> 2, n4 = T * T4;
        for (int p = lane; p < n4; p += 64) {
            const size_t q = (size_t)(ti * T + p / T4) * I + (size_t)(tj * T + 4 * (p % T4));
            float4 d[NI];
#pragma unroll
            for (int j = 0; j < NI; ++j)
                d[j] = j < ni ? load_stream(base + (size_t)j * plane + q)
                              : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if (k < nk) {
                    px(k, d[k].x, d[k + 1].x, d[k + 2].x);
                    px(k, d[k].y, d[k + 1].y, d[k + 2].y);
                    px(k, d[k].z, d[k + 1].z, d[k + 2].z);
                    px(k, d[k].w, d[k + 1].w, d[k + 2].w);
                }
            }
        }
    } else {
        for (int p = lane; p < T * T; p += 64) {
            const size_t q = (size_t)(ti * T + p / T) * I + (size_t)(tj * T + p % T);
            float d[NI];
#pragma unroll
            for (int j = 0; j < NI; ++j) d[j] = j < ni ? base[(size_t)j * plane + q] : 0.0f;
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (k < nk) px(k, d[k], d[k + 1], d[k + 2]);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        // the reduced maxima for host readers
        for (int j = 0; j < ni; ++j) meta[i0 + j].maxd_bits = md[j];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const float sk = wave_sum_f(sum[k]), mk = wave_max_f(mx[k]), rk = wave_sum_f(sr[k]);
        if (lane == 0 && k < nk) {
            const float m3 = fmaxf(__uint_as_float(md[k]), fmaxf(__uint_as_float(md[k + 1]), __uint_as_float(md[k + 2])));
            out[(size_t)(w0 + k) * un * un + tile] = tlisi_value(sk, mk, rk, m3, T);
        }
    }
}

// ------------------------------------------------------------- launchers

const char* stage_name(int st)
{
    static const char* names[kStCount] = {"reset",   "bin",   "scan",          "scatter", "grid_colfft",
                                          "row_c2r", "splat", "splat_trigger", "trigger"};
    return (st >= 0 && st < kStCount) ? names[st] : "?";
}

// Segments of a snapshot of up to n visibilities and their length: the fewest
// visibilities per thread (2, 4 or 8) that need at most 64 segments (a
// workgroup sorts 2048 visibilities in 8 to 12 us, 4096 in 16 and 8192 in 17 to
// 33, its FP64 and LDS atomics); beyond 64 * 8192 visibilities, 64 equal
// segments.
//
// Up to kOwnSums segments the merging workgroups add the offsets up themselves:
// bin and merge of three snapshots take 18.2 us with 38 segments (77777
// visibilities at 2048^2), with k_offsets between them 19.5; with 49 (100000
// at 4096^2) 27.9 and 24.3, with 64 (523776 at 8192^2) 69.8 and 58.4.
constexpr int kOwnSums = 40;
struct SegShape {
    int vpt, chunk, nseg;
};
static SegShape seg_shape(int n)
{
    constexpr int B = kBinThreads;
    SegShape q;
    q.vpt = n <= 2 * kMaxSegs * B ? 2 : (n <= 4 * kMaxSegs * B ? 4 : (n <= 8 * kMaxSegs * B ? 8 : 0));
    const int each = (n + kMaxSegs - 1) / kMaxSegs;
    q.chunk = q.vpt > 0 ? q.vpt * B : (each + B - 1) / B * B;
    q.nseg = max(1, (n + q.chunk - 1) / q.chunk);
    return q;
}

size_t bstart_words(int G) { return (size_t)boff_row(G); }

template <class VT>
static void bin_dispatch(const InputView& in, const BinView& out, int vpt, const PlanTables& p, int S, float cell,
                         double scale, const int* norm_n_dev, int norm_n_const, hipStream_t st)
{
    const dim3 grid(out.nseg + 1, S);
    const size_t lds = (size_t)(bin_keys(p.G) + 1) * sizeof(int);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kBinThreads), lds, st, in, out, norm_n_dev, norm_n_const, p.G, p.I, cell,
                           scale);
    };
    switch (vpt) {
    case 2: go(k_bin<VT, 2>); break;
    case 4: go(k_bin<VT, 4>); break;
    case 8: go(k_bin<VT, 8>); break;
    default: go(k_bin<VT, 0>); break;
    }
}

hipError_t launch_bin(const InputView& in, const WorkView& w, const PlanTables& p, int S, int nmax, float cell,
                      double scale, const int* norm_n_dev, int norm_n_const, hipStream_t st)
{
    if (p.G > kMaxGrid) return hipErrorInvalidValue;
    const SegShape q = seg_shape(nmax);
    // The segments' offsets, extents and displacements are only read by the
    // merge: they lie in each snapshot's corrected image and K tiles, which later
    // stages write (64 (g/2 + 16) ints in I^2 floats, 256 more in I (g/2 + 1)
    // pairs: I >= 64).
    const size_t plane = (size_t)p.I * p.I, tiles = (size_t)p.I * (p.M + 1) * 2;
    int* const kt = reinterpret_cast<int*>(w.kt);
    const BinView v{w.rec,  w.sorted, reinterpret_cast<int*>(w.pre), kt, kt + 256, w.bstart, w.meta, w.geom, w.pmax,
                    w.stride, plane, tiles, q.nseg, q.chunk};
    switch (in.vis_type) {
    case kVisF32: bin_dispatch<float>(in, v, q.vpt, p, S, cell, scale, norm_n_dev, norm_n_const, st); break;
    case kVisBF16: bin_dispatch<__hip_bfloat16>(in, v, q.vpt, p, S, cell, scale, norm_n_dev, norm_n_const, st); break;
    case kVisF16: bin_dispatch<__half>(in, v, q.vpt, p, S, cell, scale, norm_n_dev, norm_n_const, st); break;
    default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || q.nseg == 1) return e;
    const size_t row = (size_t)boff_row(p.G) * sizeof(int);
    if (q.nseg <= kOwnSums) {
        hipLaunchKernelGGL(k_merge<false>, dim3(q.nseg, S), dim3(kBinThreads), 2 * row, st, v, p.G);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_offsets, dim3((bin_keys(p.G) + 1 + 63) / 64, S), dim3(1024), 0, st, v, p.G);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_merge<true>, dim3(q.nseg, S), dim3(kBinThreads), row, st, v, p.G);
    return hipGetLastError();
}

template <int G, int KR>
static void stage1_dispatch(const WorkView& w, const PlanTables& p, int S, hipStream_t st)
{
    hipLaunchKernelGGL((k_stage1<G, KR>), dim3(S, G / 2 + 1), dim3(ColShape<G>::NX), 0, st, w.sorted, w.bstart, w.meta,
                       p.tw_g, w.kt, w.stride);
}

// Records per thread held in registers while a column is gridded.
template <int G>
static void stage1_pick(const WorkView& w, const PlanTables& p, int S, const Tuning& tu, hipStream_t st)
{
    if (tu.stage1_records >= 8)
        stage1_dispatch<G, 8>(w, p, S, st);
    else if (tu.stage1_records <= 2)
        stage1_dispatch<G, 2>(w, p, S, st);
    else
        stage1_dispatch<G, 4>(w, p, S, st);
}

hipError_t launch_stage1(const WorkView& w, const PlanTables& p, int S, const Tuning& tu, hipStream_t st)
{
    switch (p.G) {
    case 96: stage1_pick<96>(w, p, S, tu, st); break;
    case 192: stage1_pick<192>(w, p, S, tu, st); break;
    case 384: stage1_pick<384>(w, p, S, tu, st); break;
    case 768: stage1_pick<768>(w, p, S, tu, st); break;
    case 1536: stage1_pick<1536>(w, p, S, tu, st); break;
    case 3072: stage1_pick<3072>(w, p, S, tu, st); break;
    case 6144: stage1_pick<6144>(w, p, S, tu, st); break;
    case 12288: stage1_pick<12288>(w, p, S, tu, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int G>
static void stage2_dispatch(const WorkView& w, const PlanTables& p, int S, hipStream_t st)
{
    hipLaunchKernelGGL(k_stage2<G>, dim3(p.I / 2, S), dim3(FftPlan<G>::nt), 0, st, w.kt, w.meta, w.pmax, p.tw_g,
                       p.corr, w.pre);
}

bool row_pass_splits(int G) { return G == 12288; }

hipError_t launch_stage2(const WorkView& w, const PlanTables& p, int S, hipStream_t st)
{
    switch (p.G) {
    case 96: stage2_dispatch<96>(w, p, S, st); break;
    case 192: stage2_dispatch<192>(w, p, S, st); break;
    case 384: stage2_dispatch<384>(w, p, S, st); break;
    case 768: stage2_dispatch<768>(w, p, S, st); break;
    case 1536: stage2_dispatch<1536>(w, p, S, st); break;
    case 3072: stage2_dispatch<3072>(w, p, S, st); break;
    case 6144: stage2_dispatch<6144>(w, p, S, st); break;
    case 12288:
        hipLaunchKernelGGL(k_stage2_split<12288>, dim3(p.I / 2, S), dim3(FftPlan<6144>::nt), 0, st, w.kt, w.meta,
                           w.pmax, p.tw_m, p.wpost, p.corr, w.pre);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Two 64-pixel tiles per CU are enough to fill the GPU; with fewer, each
// workgroup's chain of loads and LDS atomics is the launch, and 32-pixel tiles
// are shorter although their borders are read twice: a call of three snapshots
// takes 33 instead of 37 us at 256^2 and 44 instead of 47 at 512^2 (2016 and 4000
// visibilities).  Batches of 4, 16, 64 and 256 snapshots at 512^2 take 57, 88,
// 198 and 710 us with 32-pixel tiles and 59, 84, 181 and 618 with 64-pixel
// ones; the lines cross at 450 to 670 of the larger tiles from 64^2 to 512^2.  From
// 1024^2 on one image has 256 of them, and a call of three takes 59 us against 63
// with the smaller ones.
int splat_tile_for(const Tuning& tu, int I, int S)
{
    if (tu.splat_tile != 0) return tu.splat_tile >= 64 ? 64 : 32;
    return I > 512 || (long)S * (I / 64) * (I / 64) >= 512 ? 64 : 32;
}

hipError_t launch_splat(const WorkView& w, const PlanTables& p, int S, const Tuning& tu, hipStream_t st)
{
    if (S <= 0) return hipSuccess;
    if (splat_tile_for(tu, p.I, S) == 64) {
        const int nt = (p.I / 64) * (p.I / 64);
        hipLaunchKernelGGL((k_splat<64, false>), dim3(nt, S), dim3(256), 0, st, w.pre, w.meta, w.geom, w.pmax, w.img,
                           p.I, 0, nullptr, nullptr, nullptr, 1);
    } else {
        const int nt = (p.I / 32) * (p.I / 32);
        hipLaunchKernelGGL((k_splat<32, false>), dim3(nt, S), dim3(256), 0, st, w.pre, w.meta, w.geom, w.pmax, w.img,
                           p.I, 0, nullptr, nullptr, nullptr, 1);
    }
    return hipGetLastError();
}

bool splat_trigger_fusable(const PlanTables& p, const Tuning& tu, int tile)
{
    // Below 4096^2 the images stay in the caches between the launches and one
    // splat over all snapshots with the trigger after it is shorter: 59 against
    // 70 us per call at 1024^2 (8128 visibilities), 105 against 108 at 2048^2
    // (32640), but 311 against 302 at 4096^2 (130816).
    return p.I >= 4096 && splat_tile_for(tu, p.I, 1) == 64 && tile == 32;
}

// The reduced trigger terms go to the K tiles' buffer, which the column and
// row passes are done with (3 floats per trigger tile; the buffer holds
// 8 I (g/2 + 1) bytes per snapshot).
static float* trigger_terms(const WorkView& w) { return reinterpret_cast<float*>(w.kt); }

hipError_t launch_splat_trigger(const WorkView& w, const PlanTables& p, int s3, const float* img_a,
                                const float* img_b, bool store, hipStream_t st)
{
    const int nt = (p.I / 64) * (p.I / 64);
    hipLaunchKernelGGL((k_splat<64, true>), dim3(nt, 1), dim3(256), 0, st, w.pre, w.meta, w.geom, w.pmax, w.img, p.I,
                       s3, img_a, img_b, trigger_terms(w), store ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_trigger_finish(const WorkView& w, const PlanTables& p, int s1, int s2, int s3, int tile, float* out,
                                 hipStream_t st)
{
    const int un = p.I / tile;
    hipLaunchKernelGGL(k_trigger_finish, dim3((un * un + 255) / 256), dim3(256), 0, st, trigger_terms(w), w.meta,
                       w.pmax, s1, s2, s3, p.I, tile, out);
    return hipGetLastError();
}

hipError_t launch_trigger(const WorkView& w, const PlanTables& p, const int* win, int nwin, int tile,
                          const TriggerOut& out, hipStream_t st)
{
    const int un = p.I / tile;
    if (un <= 0 || nwin <= 0) return hipSuccess;
    if (nwin > kMaxWindows) return hipErrorInvalidValue;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((un * un + 3) / 4, nwin), dim3(256), 0, st, w.img, w.meta, w.pmax, win, p.I,
                           tile, out);
    };
    if (tile % 4 == 0)
        go(k_trigger<kTrigWide>);
    else if (tile * tile > 128)
        go(k_trigger<kTrigDeep>);
    else
        go(k_trigger<kTrigSmall>);
    return hipGetLastError();
}

hipError_t launch_trigger_run(const WorkView& w, const PlanTables& p, int s0, int nwin, int tile, float* out,
                              hipStream_t st)
{
    const int un = p.I / tile;
    if (un <= 0 || nwin <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_trigger_run, dim3((un * un + 3) / 4, (nwin + kRunWin - 1) / kRunWin), dim3(256), 0, st,
                       w.img, w.meta, w.pmax, s0, nwin, p.I, tile, out);
    return hipGetLastError();
}

// One wave per snapshot: the slot maxima into meta.
__global__ __launch_bounds__(64) void k_max_finalize(SnapMeta* __restrict__ meta, unsigned* __restrict__ pmax)
{
    const int s = blockIdx.x, lane = threadIdx.x;
    const unsigned mp = wave_max_u(*max_slot(pmax, s, 0, lane));
    const unsigned md = wave_max_u(*max_slot(pmax, s, 1, lane));
    if (lane == 0) {
        meta[s].maxp_bits = mp;
        meta[s].maxd_bits = md;
    }
}

hipError_t launch_max_finalize(const WorkView& w, int S, hipStream_t st)
{
    if (S <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_max_finalize, dim3(S), dim3(64), 0, st, w.meta, w.pmax);
    return hipGetLastError();
}

// ------------------------------------------------------------ FFT check

template <int N>
__global__ __launch_bounds__(FftPlan<N>::nt) void k_fft_check(float2* __restrict__ data, const float2* __restrict__ tw)
{
    constexpr int NT = FftPlan<N>::nt;
    __shared__ float2 fb[lds_len(N)];
    float2* d = data + (size_t)blockIdx.x * N;
    for (int i = threadIdx.x; i < N; i += NT) fb[lds_pad(i)] = d[i];
    __syncthreads();
    fft_inverse<N>(fb, tw, threadIdx.x);
    for (int i = threadIdx.x; i < N; i += NT) d[i] = fb[lds_pad(i)];
}

hipError_t launch_fft_check(int n, float2* data, const float2* tw, int count, hipStream_t st)
{
    switch (n) {
#define FIP_FFT_CASE(N_)                                                                                  \
    case N_:                                                                                              \
        hipLaunchKernelGGL(k_fft_check<N_>, dim3(count), dim3(FftPlan<N_>::nt), 0, st, data, tw);        \
        break;
        FIP_FFT_CASE(48)
        FIP_FFT_CASE(96)
        FIP_FFT_CASE(192)
        FIP_FFT_CASE(384)
        FIP_FFT_CASE(768)
        FIP_FFT_CASE(1536)
        FIP_FFT_CASE(3072)
        FIP_FFT_CASE(6144)
        FIP_FFT_CASE(12288)
#undef FIP_FFT_CASE
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ----------------------------------------------------- plan-side helpers

template <int N>
static void twiddles_for(float2* out)
{
    using P = FftPlan<N>;
    int ns = 1, off = 0;
    for (int s = 0; s < P::nstages; ++s) {
        const int R = P::radix[s];
        if (ns > 1) {
            for (int r = 1; r < R; ++r) {
                for (int k = 0; k < ns; ++k) {
                    // exp(+2 pi i r k / (ns R)), argument reduced exactly in integers
                    const long long num = (long long)r * k % ((long long)ns * R);
                    const double ang = 2.0 * M_PI * (double)num / (double)(ns * R);
                    out[off + (r - 1) * ns + k] = make_float2((float)cos(ang), (float)sin(ang));
                }
            }
            off += (R - 1) * ns;
        }
        ns *= R;
    }
}

bool fft_size_supported(int n)
{
    switch (n) {
    case 48: case 96: case 192: case 384: case 768: case 1536: case 3072: case 6144: case 12288:
        return true;
    default:
        return false;
    }
}

void make_stage_twiddles(int n, float2* out)
{
    switch (n) {
    case 48: twiddles_for<48>(out); break;
    case 96: twiddles_for<96>(out); break;
    case 192: twiddles_for<192>(out); break;
    case 384: twiddles_for<384>(out); break;
    case 768: twiddles_for<768>(out); break;
    case 1536: twiddles_for<1536>(out); break;
    case 3072: twiddles_for<3072>(out); break;
    case 6144: twiddles_for<6144>(out); break;
    case 12288: twiddles_for<12288>(out); break;
    default: break;
    }
}

int fft_threads(int n)
{
    switch (n) {
    case 48: return FftPlan<48>::nt;
    case 96: return FftPlan<96>::nt;
    case 192: return FftPlan<192>::nt;
    case 384: return FftPlan<384>::nt;
    case 768: return FftPlan<768>::nt;
    case 1536: return FftPlan<1536>::nt;
    case 3072: return FftPlan<3072>::nt;
    case 6144: return FftPlan<6144>::nt;
    case 12288: return FftPlan<12288>::nt;
    default: return 0;
    }
}

}  // namespace fip
