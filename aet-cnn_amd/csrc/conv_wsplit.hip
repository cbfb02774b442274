// Weight gradient of 3x3 stride-1 convolutions with padding 1:
// dW[f][c][ki][kj] = sum over images and positions of
// dy[f][oy][ox] * x[c][oy+ki-1][ox+kj-1], on the bf16 matrix cores with
// three exact bf16 pieces per float (the arithmetic of conv_split.hip).
//
// The contraction runs over positions, which are contiguous in both tensors,
// so an operand fragment (8 consecutive positions of one row of f or c) is a
// 16-byte LDS read and a tap's kj is a shift of x by whole elements.  A K
// step is one input row y of a unit: 16 positions as two segments of 8,
// either adjacent columns of one image or, when the row has an odd number of
// segments, the same segment of two images.  At a step a wave reads x's row
// once, forms its three shifted versions in registers (a segment keeps its
// neighbour on each side beside it) and multiplies them with the dy rows
// y-ki+1 of a ring in LDS: one x row and one dy row are split and staged per
// step for nine taps of MFMAs.  Rows of consecutive units follow each other
// in the ring, so a slice is any range of steps.
//
// A workgroup is 64 filters x 64 channels x 9 taps: two groups of four waves
// take halves of a slice's steps, each wave 32 x 32 x 9 (144 accumulator
// registers), and add their sums in LDS, which halves the partial sums
// written per CU.  A step's staging is spread over all lanes (each one
// segment of one row, loaded a step ahead, split beside the MFMAs); dy rows
// outside the image are read from a row of zeros, so a step has no branch.
//
// Bound: the matrix pipe beside the staging and the additions; 2.3 us per step
// of 54 MFMAs on each of two waves per SIMD (1.44 us at the full clock).
// Measured with the reduction, batch 128, fp32 kernel before -> now: 128 -> 128 @
// 32x32 286 -> 184 us (210 TFLOP/s), 512 -> 512 @ 8x8 292 -> 184, 384 -> 384 @
// 13x13 461 -> 336 (rows of 13 of 16 positions); batch 32, 512 -> 512 @ 8x8 86 ->
// 64.
// Non-finite sums are computed again as in conv_split.hip: with NaNs
// everywhere the first of these takes 920 us (310 on the fp32 kernel).  What
// the recomputation keeps in registers is counted beside the loop's: written
// with indexed sums it made the kernel spill 82 registers after the loop
// (188 us instead of 183, 62.9 MB written a launch instead of 37.7).
// Error against 64 bits, batch 128: 128 -> 128 @ 32x32 2.5e-7 (fp32 kernel
// 8.2e-7; 7.7e-7 with one accumulator for all products, 5% faster),
// 384 -> 384 @ 13x13 3.1e-7 (7.8e-7; 7.2e-7), batch 8, 64 -> 64 @ 112x112
// 1.9e-7 (2.5e-7; 3.8e-7).
// Partial sums laid out [tap][f][c], 32 channels a line: stored as dw is
// ([f][c][tap], 36 bytes between lanes) the first of these took 237 us.
#include "conv_wsplit.hpp"
#include "pieces.hpp"

namespace ach {

struct Wsplit {
    const float *x, *dy;
    float *part;
    int B, C, H, W, F;
    int S;         // steps: units * H
    int spw;       // steps per group
    int pair;      // the two segments are of two images
    int nu;        // units per image (pair)
    int cols;      // columns per unit
    int mt, ct, tiles;
    FastDiv dh, dnu;
};

// W8: rows of a multiple of 8 positions (whole segments, 16-byte loads)
template <bool W8>
__global__ void __launch_bounds__(512, 2) k_conv_wsplit(Wsplit p)
{
    constexpr int KS = 3, P = 1, NT = 256, T = KS * KS;
    constexpr int R = 64;                      // rows of dy (f) and of x (c) per workgroup
    constexpr int ROWB = 6 * R * 16;           // bytes of a staged row: [piece][seg][r] x 16
    constexpr int NBB = 6 * R * 4;             // its neighbours: [piece][seg][r] x (right, left)
    constexpr int NR = KS + 1;                 // dy rows in the ring
    constexpr int GB = (NR + 1) * ROWB + 2 * (ROWB + NBB) + NBB;
    extern __shared__ __align__(16) char smem[];
    const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT);
    const int tid = (int)threadIdx.x - grp * NT;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wf = wave & 1, wc = wave >> 1;
    const int half = lane >> 5, l32 = lane & 31;
    // a group's stages: the dy ring, a row of zeros, two x rows with their
    // neighbours, a spare neighbour block
    char *const dyb = smem + grp * GB, *const zero = dyb + NR * ROWB;
    char *const xb = zero + ROWB;

    // XCD x runs a contiguous range of (slice, tile) pairs, tiles fastest: the
    // tiles of a slice share its rows of x and dy in that XCD's L2
    int id = blockIdx.x + blockIdx.y * gridDim.x;
    {
        const int G = gridDim.x * gridDim.y, g8 = G >> 3, r8 = G & 7, xcd = id & 7, k = id >> 3;
        id = xcd * g8 + min(xcd, r8) + k;
    }
    const int z = id / p.tiles;
    id -= z * p.tiles;
    const int c0 = (id % p.ct) * R, m0 = (id / p.ct) * R;
    const int s0 = min(p.S, (z * 2 + grp) * p.spw), s1 = min(p.S, s0 + p.spw);
    const int HW = p.H * p.W;

    // Staging: waves 0 and 1 take 32 rows of dy each, 2 and 3 of x; a lane one
    // segment (8 positions) of one row, and for x the position on each side
    // of it.  A wave's role is a matter of operands, not of branches.
    const bool isx = wave >= 2;
    const int trow = (wave & 1) * 32 + (lane >> 1), seg = lane & 1;
    const int nrow = isx ? p.C : p.F, row = (isx ? c0 : m0) + trow;
    const __amdgpu_buffer_rsrc_t rs =
        make_rsrc(isx ? p.x : p.dy, (unsigned)((size_t)p.B * nrow * HW * 4));
    // (readfirstlane hides the role from the optimiser, which would turn the
    // loop body into a branch per role)
    auto role = [&](int x, int d) { return __builtin_amdgcn_readfirstlane(isx ? x : d); };
    const int lead = role(0, P);  // step s brings x row s and dy row s + P
    const int slot0 = role((NR + 1) * ROWB, 0), slotm = role(1, NR - 1);
    const int slotb = role(ROWB + NBB, ROWB), slotn = role(0, P + NR);
    const int nb0 = role((NR + 2) * ROWB, (NR + 3) * ROWB + 2 * NBB), nbb = role(ROWB + NBB, 0);
    const int side = role(0, (int)kOOB);
    const int ps = p.pair ? 1 : 0, segc = ps ? 0 : seg * 8, segb = ps ? seg : 0;
    const int lanebase = (row + segb * nrow) * HW + segc;
    char *const st0 = dyb + (trow + seg * R) * 16;
    char *const st1 = dyb + (seg * R + trow) * 4;
    auto load = [&](int s, float *r) {
        const int ds = s + lead, dc = max(ds, 0);
        const int u = fdiv(dc, p.dh), y = dc - u * p.H, q = fdiv(u, p.dnu);
        const int cu = (u - q * p.nu) * p.cols, b0 = q << ps;
        const int rows = (unsigned)ds < (unsigned)p.S ? nrow : 0;
        const int col = cu + segc, left = p.W - col;
        const bool ok = (row < rows) & (b0 + segb < p.B);
        const int base = (lanebase + b0 * nrow * HW + y * p.W + cu) * 4;
        if constexpr (W8) {
            const int o = (ok & (left > 0)) ? base : (int)kOOB;
            const float4 a = bload4_so(rs, o, 0), b = bload4_so(rs, o, 16);
            r[0] = a.x; r[1] = a.y; r[2] = a.z; r[3] = a.w;
            r[4] = b.x; r[5] = b.y; r[6] = b.z; r[7] = b.w;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) r[j] = bload(rs, (ok & (left > j)) ? base + 4 * j : (int)kOOB);
        }
        // the neighbours (a dy row has none: out-of-range offsets)
        r[8] = bload(rs, ((ok & (left > 8)) ? base + 32 : (int)kOOB) | side);
        r[9] = bload(rs, ((ok & (col > 0) & (left > -1)) ? base - 4 : (int)kOOB) | side);
    };
    auto store = [&](int s, const float *r) {
        v4u pc[3];
        split8(r, pc);
        const int slot = (s + slotn) & slotm;
        char *const dst = st0 + slot0 + slot * slotb;
        unsigned *const nb = reinterpret_cast<unsigned *>(st1 + nb0 + slot * nbb);
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<v4u *>(dst + q * 2 * R * 16) = pc[q];
        const float a = r[8] * kPieceUp, b = r[9] * kPieceUp;
        const unsigned h = pk_bf16(a, b);
        const float ra = a - bf_lo(h), rb = b - bf_hi(h);
        const unsigned m = pk_bf16(ra, rb);
        nb[0] = h;
        nb[2 * R] = m;
        nb[4 * R] = pk_bf16(ra - bf_lo(m), rb - bf_hi(m));
    };

    v16f acc[KS][KS];
#pragma unroll
    for (int i = 0; i < KS; ++i)
#pragma unroll
        for (int j = 0; j < KS; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    for (int i = tid * 16; i < ROWB; i += NT * 16) *reinterpret_cast<v4u *>(zero + i) = v4u{0, 0, 0, 0};
    // steps s0-2 and s0-1 bring the ring's first dy rows (their x rows go to
    // slots that later steps overwrite)
    float r[10];
    {
        float r0[10], r1[10], r2[10];
        load(s0 - 2, r0);
        load(s0 - 1, r1);
        load(s0, r2);
        load(s0 + 1, r);
        store(s0 - 2, r0);
        store(s0 - 1, r1);
        store(s0, r2);
    }
    __syncthreads();
    // every group runs p.spw iterations, one past its last step on rows that
    // read as zero
    int y = s0 - fdiv(s0, p.dh) * p.H;
    const v16f none = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const unsigned frag = (half * R + l32) * 16;
    for (int s = s0; s < s0 + p.spw; ++s) {
        const char *const xr = xb + (s & 1) * (ROWB + NBB);
        v4u u[3], a[2][3];
        unsigned nb[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            u[q] = *reinterpret_cast<const v4u *>(xr + frag + (q * 2 * R + wc * 32) * 16);
            nb[q] = reinterpret_cast<const unsigned *>(xr + ROWB)[(q * 2 + half) * R + wc * 32 + l32];
        }
        // tap ki reads dy row y - ki + P, or zeros beyond the image (and past
        // the slice's end)
        const unsigned live = s < s1 ? (unsigned)p.H : 0u;
        auto load_a = [&](int i) {
            const int slot = ((s - i + P + NR) & (NR - 1)) * ROWB;
            const int in = -(int)((unsigned)(y - i + P) < live);  // all ones or zero
            const char *const dr = dyb + ((slot & in) | (NR * ROWB & ~in));
#pragma unroll
            for (int q = 0; q < 3; ++q)
                a[i & 1][q] = *reinterpret_cast<const v4u *>(dr + frag + (q * 2 * R + wf * 32) * 16);
        };
        load_a(0);
        v4u b[KS][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const v4u v = u[q];
            const unsigned m0_ = __builtin_amdgcn_alignbit(v[1], v[0], 16);
            const unsigned m1_ = __builtin_amdgcn_alignbit(v[2], v[1], 16);
            const unsigned m2_ = __builtin_amdgcn_alignbit(v[3], v[2], 16);
            b[0][q] = v4u{__builtin_amdgcn_alignbit(v[0], nb[q], 16), m0_, m1_, m2_};
            b[1][q] = v;
            b[2][q] = v4u{m0_, m1_, m2_, __builtin_amdgcn_alignbit(nb[q], v[3], 16)};
        }
        // the rows of step s + 1, loaded a step ago, are split and stored and
        // those of step s + 2 loaded beside the MFMAs
        store(s + 1, r);
        load(s + 2, r);
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            if (i + 1 < KS) load_a(i + 1);
            const v4u *ca = a[i & 1];
            // The matrix unit cuts off what it aligns to the largest term of a
            // sum: with all six products added to the accumulator the sums
            // were low by 3e-7 to 7e-7 of their size on long contractions.
            // The five small products are summed from zero and added once.
#pragma unroll
            for (int j = 0; j < KS; ++j) {
                v16f t = MFMA_BF(as_bf(ca[2]), as_bf(b[j][0]), none);
                t = MFMA_BF(as_bf(ca[0]), as_bf(b[j][2]), t);
                t = MFMA_BF(as_bf(ca[1]), as_bf(b[j][1]), t);
                t = MFMA_BF(as_bf(ca[1]), as_bf(b[j][0]), t);
                acc[i][j] = MFMA_BF(as_bf(ca[0]), as_bf(b[j][0]), acc[i][j]);
                acc[i][j] += MFMA_BF(as_bf(ca[0]), as_bf(b[j][1]), t);
            }
        }
        if (++y == p.H) y = 0;
        __syncthreads();
    }

    bool bad = false;
#pragma unroll
    for (int q = 0; q < T; ++q)
#pragma unroll
        for (int e = 0; e < 16; ++e) bad |= !(fabsf(acc[q / KS][q % KS][e]) <= 3.402823466e38f);
    const int c = c0 + wc * 32 + l32, f = m0 + wf * 32 + 4 * half;
    float down = kSumDown;
    if (__ballot(bad)) {  // this wave's tiles again on the fp32 instructions
        down = 1.f;
#pragma unroll
        for (int q = 0; q < T; ++q)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[q / KS][q % KS][e] = 0.f;
        const int fr = m0 + wf * 32 + l32;
        const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, (unsigned)((size_t)p.B * p.C * HW * 4));
        const __amdgpu_buffer_rsrc_t rd = make_rsrc(p.dy, (unsigned)((size_t)p.B * p.F * HW * 4));
#pragma unroll
        for (int i = 0; i < KS; ++i) {
#pragma unroll 1
            for (int s = s0; s < s1; ++s) {  // lane half h: segment h
                const int un = fdiv(s, p.dh), iy = s - un * p.H, q = fdiv(un, p.dnu);
                const int cb = (un - q * p.nu) * p.cols, b = (q << ps) + (ps ? half : 0);
                const int ox0 = cb + (ps ? 0 : half * 8);
                const bool okf = (fr < p.F) & (b < p.B), okc = (c < p.C) & (b < p.B);
                const int xrow = (b * p.C + c) * HW + iy * p.W, drow = (b * p.F + fr) * HW;
                // t = 1: the dy row that this tap row meets beyond x's first
                // or last row, with that row of x (products with padding
                // zeros, which no step forms)
                const int edge = (iy == 0 && i < P) || (iy == p.H - 1 && i > P);
#pragma unroll 1
                for (int t = 0; t <= edge; ++t) {
                    const int oy = t ? iy : iy - i + P;
                    if (oy < 0 || oy >= p.H) continue;
                    float dv[8], xv[10];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        dv[e] = bload(rd, boff(okf & (ox0 + e < p.W), drow + oy * p.W + ox0 + e));
#pragma unroll
                    for (int e = 0; e < 10; ++e)
                        xv[e] = bload(rx, boff(okc & !t & ((unsigned)(ox0 + e - P) < (unsigned)p.W),
                                               xrow + ox0 + e - P));
                    // a row's sums stand by themselves, as one chain over the
                    // slice had more error than the fp32 kernel's shorter ones
                    v16f sum[KS];
#pragma unroll
                    for (int j = 0; j < KS; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r) sum[j][r] = 0.f;
                    // (a position past the row's end meets no x: its zero
                    // delta must not meet an infinite one)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
#pragma unroll
                        for (int j = 0; j < KS; ++j)
                            sum[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                dv[e], ox0 + e < p.W ? xv[e + j] : 0.f, sum[j], 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < KS; ++j) acc[i][j] += sum[j];
                }
            }
        }
    }
    // the groups exchange tiles in rounds of QR taps: group q & 1 stores tap q
    constexpr int QR = 4;
    float4 *const xs = reinterpret_cast<float4 *>(smem);
#pragma unroll
    for (int q0 = 0; q0 < T; q0 += QR) {
        if (q0) __syncthreads();
#pragma unroll
        for (int q = q0; q < (q0 + QR < T ? q0 + QR : T); ++q)
            if ((q & 1) != grp) {
                const v16f t = acc[q / KS][q % KS] * down;
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4)
                    xs[((q - q0) * 4 + r4) * NT + tid] =
                        make_float4(t[4 * r4], t[4 * r4 + 1], t[4 * r4 + 2], t[4 * r4 + 3]);
            }
        __syncthreads();
#pragma unroll
        for (int q = q0; q < (q0 + QR < T ? q0 + QR : T); ++q)
            if ((q & 1) == grp) {
                const v16f t = acc[q / KS][q % KS] * down;
                const int ld = p.C;
                float *base = p.part + (((size_t)z * T + q) * p.F + f) * ld + c;
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    const float4 o = xs[((q - q0) * 4 + r4) * NT + tid];
                    const float v[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (c < p.C && f + 8 * r4 + e < p.F)
                            base[(size_t)(8 * r4 + e) * ld] = t[4 * r4 + e] + v[e];
                }
            }
    }
}

// dw[f][c][t] += sum over z of part[z][t][f][c], z ascending within quarters
// of the slices and the quarters' sums in order, then the SGD step when sg.w.
// A block takes 64 channels of one filter: its four waves sum a quarter of
// the slices each (64 consecutive channels per load), and the 64 x 9 results
// are consecutive in dw.
__global__ void __launch_bounds__(256) k_wsplit_reduce(const float *__restrict__ part,
                                                       float *__restrict__ dw, int F, int C,
                                                       int splits, Sgd sg)
{
    constexpr int T = 9;
    __shared__ float sums[4][64][T];
    const int f = blockIdx.y, c0 = blockIdx.x * 64;
    const int lane = threadIdx.x & 63, zq = threadIdx.x >> 6, c = c0 + lane;
    const int zs = (splits + 3) / 4, z0 = min(splits, zq * zs), z1 = min(splits, z0 + zs);
    if (c < C) {
        const size_t zstep = (size_t)T * F * C, tstep = (size_t)F * C;
        const float *p = part + (size_t)f * C + c;
        float s[T];
#pragma unroll
        for (int t = 0; t < T; ++t) s[t] = 0.f;
        int z = z0;
        for (; z + 2 <= z1; z += 2) {
            float v[2][T];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int t = 0; t < T; ++t) v[u][t] = p[(z + u) * zstep + t * tstep];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int t = 0; t < T; ++t) s[t] += v[u][t];
        }
        if (z < z1) {
#pragma unroll
            for (int t = 0; t < T; ++t) s[t] += p[z * zstep + t * tstep];
        }
#pragma unroll
        for (int t = 0; t < T; ++t) sums[zq][lane][t] = s[t];
    }
    __syncthreads();
    const int n = min(64, C - c0) * T;
    float *d = dw + ((size_t)f * C + c0) * T;
    float *w = sg.w ? sg.w + ((size_t)f * C + c0) * T : nullptr;
    const float *q = &sums[0][0][0];
    for (int i = threadIdx.x; i < n; i += 256) {
        float o = d[i] + (((q[i] + q[64 * T + i]) + q[128 * T + i]) + q[192 * T + i]);
        if (w) {
            float a = w[i];
            sgd_step(a, o, sg.dc, sg.lc, sg.mom);
            w[i] = a;
        }
        d[i] = o;
    }
}

int wsplit_reduce(const ConvGeom &g, const WsplitPlan &pl, const float *part, float *dw,
                  const Sgd &sg, hipStream_t st)
{
    hipLaunchKernelGGL(k_wsplit_reduce, dim3((g.C + 63) / 64, g.F), dim3(256), 0, st, part, dw, g.F,
                       g.C, pl.splits, sg);
    return check_launch();
}

static int wsplit_go(Wsplit &p, const WsplitPlan &pl, hipStream_t st)
{
    constexpr int R = 64, ROWB = 6 * R * 16, NBB = 6 * R * 4;
    p.mt = (p.F + R - 1) / R;
    p.ct = (p.C + R - 1) / R;
    p.tiles = p.mt * p.ct;
    const size_t lds = 2 * (size_t)(5 * ROWB + 2 * (ROWB + NBB) + NBB);
    auto kern = p.W % 8 == 0 ? &k_conv_wsplit<true> : &k_conv_wsplit<false>;
    const int rc = check(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    if (rc) return rc;
    hipLaunchKernelGGL(kern, dim3(p.tiles, pl.splits), dim3(512), lds, st, p);
    return check_launch();
}

// units per image (pair), columns per unit and whether segments pair images
static void wsplit_units(const ConvGeom &g, int &pair, int &nu, int &cols, long long &units)
{
    const int segs = (g.W + 7) / 8;
    pair = (segs & 1) && g.B > 1;
    nu = pair ? segs : (segs + 1) / 2;
    cols = pair ? 8 : 16;
    units = (long long)(pair ? (g.B + 1) / 2 : g.B) * nu;
}

// 119 steps, 384 -> 384 @ 13x13: 3.1e-7, after a relu 2.7e-7.  (349 -> 463 @
// 43x43, batch 10, in groups of 129 steps was at 3.4e-7, the fp32 kernel, whose
// parts are of 144 products, at 2.5e-7.)
constexpr StepError kStepError = {2.55, 2.2};

WsplitPlan wsplit_plan(const ConvGeom &g, const Fp32Wgrad &fp32, int room)
{
    WsplitPlan pl{};
    if (g.S != 1 || g.KS != 3 || 2 * g.P != g.KS - 1 || g.OH != g.H || g.OW != g.W) return pl;
    int pair, nu, cols;
    long long units;
    wsplit_units(g, pair, nu, cols, units);
    const long long S = units * g.H;
    if (S >= (1ll << 26)) return pl;
    const long long tiles = (long long)((g.F + 63) / 64) * ((g.C + 63) / 64);
    // Time model (us), fitted to 185 of 900 layer shapes that run here: a step
    // of the two groups' eight waves, 2.1-2.4 where rows are whole segments,
    // 2.5-2.9 where they are not, 3.3-4.5 and 4.0-5.4 where, besides, a line of
    // memory holds three or five segments of an image pair, which are read far
    // apart (the line comes from HBM for each); the partial sums written and
    // read; and prologue, exchange and reduction.
    const double step = g.W % 8 == 0 ? 2.4 : !pair || nu < 3 ? 2.8 : nu < 5 ? 4.2 : 4.8;
    const double mn4 = (double)g.F * g.C * g.KS * g.KS * 4;
    const double limit = 0.95 * fp32.us;
    if (limit < 12.0 + 4 * step + 4.0) return pl;  // the shortest plan is no faster
    auto precise = [&](int s, long long spw) {
        return no_more_error(kStepError, (double)spw, s / 4.0 + 4,
                             (double)g.B * g.H * g.W / fp32.parts, fp32.adds);
    };
    double best = -1;
    for (int k = 1; k <= 10; ++k) {  // one to six rounds of 256 workgroups, or a part of one
        const int s = k <= 6 ? (int)(256 * k / tiles) : (int)(256 / ((k - 5) * tiles));
        if (s < 1 || s > room) continue;
        const long long spw = (S + 2 * s - 1) / (2 * s);
        if (!precise(s, spw) || (s > 1 && spw < 4)) continue;
        const long long rounds = (tiles * s + 255) / 256;
        const double t = 12.0 + rounds * (spw * step + 4.0) + s * mn4 * 2 / 5e6;
        if (best < 0 || t < best * 0.995) {
            best = t;
            pl.splits = s;
            pl.spw = (int)spw;
        }
    }
    if (best < 0 && room >= 1 && precise(1, (S + 1) / 2)) {  // more tiles than fill the chip
        pl.splits = 1;
        pl.spw = (int)((S + 1) / 2);
        best = 12.0 + (tiles + 255) / 256 * (pl.spw * step + 4.0) + mn4 * 2 / 5e6;
    }
    pl.ok = best >= 0 && best < limit;
    return pl;
}

int wsplit_launch(const ConvGeom &g, const WsplitPlan &pl, const float *x, const float *dy,
                  float *part, hipStream_t st)
{
    Wsplit p{};
    p.x = x; p.dy = dy; p.part = part;
    p.B = g.B; p.C = g.C; p.H = g.H; p.W = g.W; p.F = g.F;
    long long units;
    wsplit_units(g, p.pair, p.nu, p.cols, units);
    p.S = (int)(units * g.H);
    p.spw = pl.spw;
    p.dh = make_fastdiv((unsigned)g.H);
    p.dnu = make_fastdiv((unsigned)p.nu);
    return wsplit_go(p, pl, st);
}

}  // namespace ach
