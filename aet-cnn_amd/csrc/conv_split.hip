// Convolution GEMMs on the bf16 matrix cores with exact three-piece operands.
//
// A finite float is the sum of three bf16 values (8 significant bits each,
// rounded to nearest, the residuals exact): a = a0 + a1 + a2 with
// |a1| <= 2^-8 |a|, |a2| <= 2^-17 |a| (about).  A product a*b is taken as the
// six piece products down to 2^-17 relative (a0b0, a0b1, a1b0, a1b1, a0b2,
// a2b0); each is exact in the matrix unit, and what is left out (a1b2, a2b1,
// a2b2) is below 2^-24 |ab|, what rounding an fp32 product can lose.  v_mfma_f32_32x32x16_bf16 adds 16 such products to the fp32
// accumulator at once, where v_mfma_f32_32x32x2_f32 adds two, and runs 16
// times its rate, so the six passes cost 6/16 of the fp32 instruction's matrix
// time and the sums round an eighth as often.
//
// Non-finite values: an infinity (or a finite value above 2^103, which the
// operands' scale of 2^24 takes to one) leaves non-finite residuals, so the
// tile's sums come out non-finite; a wave that finds a non-finite sum
// computes its tile again on the fp32 instructions, straight from memory,
// which gives the infinities and NaNs of fp32 arithmetic (and, a channel
// chunk's sums standing by themselves, no more error than the fp32 kernels:
// 2.2e-7 against 6.0e-7 for 128 -> 128 @ 32x32 at 1e35).  With NaNs
// everywhere that layer takes 560 us, 172 without and 310 on the fp32 kernel;
// one NaN in the batch takes it to 240.
//
// The workgroup: four waves of 32 filters x 128 positions (2 x 64 or 1 x 32
// for 33-64 or up to 32 filters).  A chunk of 16 input channels of the tile's
// patch (its rows with their halo) is split once and staged in LDS pixel by
// pixel, [3 pieces][16 channels], so a tap's operand is one aligned 16-byte
// read per piece at a uniform offset: every value is split once per chunk
// instead of once per tap, and 9 (25) taps of MFMAs run between barriers.
// The filter rows go straight from memory to registers and are split there
// (44 VALU per 24 MFMAs, in the matrix pipe's shadow).
// The products below the leading one have an accumulator of their own, so
// the large sums round once per 16 products: the error against 64 bits is
// 0.36 of the fp32 instruction's (2.2e-7 against 6.0e-7, 128 -> 128 @ 32x32).
//
// Bound: the matrix pipe at the clock that six bf16 passes sustain.  The same
// loop without loads, splits and LDS runs 276 TFLOP/s (fp32-equivalent),
// the kernel 221-222 where the fp32 kernel ran 138-142 (3x3, batch 128: 128 ->
// 128 @ 32x32 272 -> 175 us, 384 -> 384 @ 13x13 416 -> 259 us), and 214-233
// against 131 on 5x5 filters (96 -> 256 @ 27x27 872 -> 493 us); without the
// filter loads and without LDS reads 12% and 9% less.
#include "conv_split.hpp"
#include "pieces.hpp"

namespace ach {

// ---------------------------------------------------------------------------
constexpr int SP_CH = 16;     // input channels per chunk (one MFMA K)
constexpr int SP_PXB = 112;   // LDS bytes per patch pixel: 3 pieces x 16 channels, padded so
                              // that eight consecutive pixels' 16-byte reads hit all banks
constexpr int SP_BN = 128;    // output positions per workgroup
constexpr int SP_LDS = 160 * 1024;  // LDS of a CU

struct SplitFwd {
    const float *x, *wt;
    float *y, *part;
    int B, C, H, W, M, P, OH, OW, N;
    int VH, PW;           // padded rows per image, padded columns
    int nchunk, cps;      // channel chunks, chunks per (slice, group)
    int splits, nbuf, npx;
    int mt, tiles;
    FastDiv dohw, dow, dh, dw;
    Epi e;
};

template <int WM, int WN, int KG, int KS, int TPT, bool EPI>
__global__ void __launch_bounds__(64 * WM * WN * KG, 2) k_conv_split(SplitFwd p)
{
    constexpr int NT = 64 * WM * WN, NF = 4 / WN, T = KS * KS;
    extern __shared__ __align__(16) char smem[];
    const int grp = KG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT) : 0;
    const int tid = (int)threadIdx.x - grp * NT;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int half = lane >> 5, l32 = lane & 31;

    // XCD x runs the contiguous logical tiles [x*G/8, (x+1)*G/8), M fastest:
    // the M tiles of one patch share that XCD's L2
    int id = blockIdx.x;
    {
        const int g8 = p.tiles >> 3, r8 = p.tiles & 7, xcd = id & 7, k = id >> 3;
        id = xcd * g8 + min(xcd, r8) + k;
    }
    const int nt = id / p.mt, n0 = nt * SP_BN, m0 = (id - nt * p.mt) * 32 * WM;
    const int z = blockIdx.y;
    const int ch0 = (z * KG + grp) * p.cps;
    const int ch1 = min(p.nchunk, ch0 + p.cps);
    const int HW = p.H * p.W, OHW = p.OH * p.OW;

    // The tile's patch in LDS: the virtual rows [vs, ve] of the stack of
    // padded images.  Its padding is zeroed once; the staging tasks of a chunk
    // are the (pixel, channel half) pairs of the input rows [g0, g1] (rows of
    // the image stack b*H + r), consecutive lanes on consecutive pixels.
    int vs, npx, g0, nreal;
    {
        const int b0 = fdiv(n0, p.dohw), oh0 = fdiv(n0 - b0 * OHW, p.dow);
        const int nl = min(n0 + SP_BN, p.N) - 1;
        const int b1 = fdiv(nl, p.dohw), oh1 = fdiv(nl - b1 * OHW, p.dow);
        vs = b0 * p.VH + oh0;
        npx = (b1 * p.VH + oh1 + KS - vs) * p.PW;
        g0 = b0 * p.H + min(max(oh0 - p.P, 0), p.H);
        nreal = (b1 * p.H + min(max(oh1 - p.P + KS, 0), p.H) - g0) * p.W;
    }
    unsigned voff[TPT];
    int loff[TPT];
#pragma unroll
    for (int i = 0; i < TPT; ++i) {
        const int q = tid + NT * i;
        const int hf = q >= nreal ? 1 : 0, px = q - hf * nreal;
        const int r = fdiv(px, p.dw), cc = px - r * p.W;
        const int b = fdiv(g0 + r, p.dh), rr = g0 + r - b * p.H;
        const int at = (b * p.VH + rr + p.P - vs) * p.PW + cc + p.P;
        // (rows or columns that no window reads, with a padding wider than
        // the window, go to the spare slot after the patch)
        const bool ok = px < nreal && at >= 0 && at < npx && cc + p.P < p.PW && rr + p.P < p.VH;
        voff[i] = ok ? (unsigned)((b * p.C + hf * 8) * HW + rr * p.W + cc) * 4u : kOOB;
        loff[i] = ok ? at * SP_PXB + hf * 16 : p.npx * SP_PXB;
    }
    const int bufb = (p.npx + 1) * SP_PXB;
    char *const stage = smem + (size_t)grp * p.nbuf * bufb;
    // A chunk's loads go through a descriptor moved to the chunk (and tap),
    // so the scalar offsets of its eight channels are loop-invariant.  The
    // last chunk of a C that is not a multiple of 16 ends at channel C: its
    // first channels, which the chunk before it holds too, are staged as zero.
    auto chan0 = [&](int ch) { return min(ch * SP_CH, p.C - SP_CH); };
    const unsigned xbytes = (unsigned)((size_t)p.B * p.C * HW * 4);
    const unsigned wbytes = (unsigned)((size_t)p.C * T * p.M * 4);
    for (int i = tid * 16; i < p.nbuf * bufb; i += NT * 16)
        *reinterpret_cast<v4u *>(stage + i) = v4u{0, 0, 0, 0};
    __syncthreads();
    float sv[TPT][8];
    auto load_px = [&](int ch) {
        const int c0 = chan0(ch), dup = ch * SP_CH - c0;
        const unsigned d = (unsigned)c0 * (unsigned)HW * 4u;
        const __amdgpu_buffer_rsrc_t rx =
            make_rsrc(reinterpret_cast<const char *>(p.x) + d, xbytes - d);
#pragma unroll
        for (int i = 0; i < TPT; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) sv[i][j] = bload_so(rx, voff[i], (unsigned)(j * HW) * 4u);
        if (dup) {
#pragma unroll
            for (int i = 0; i < TPT; ++i) {
                const int mine = dup - (tid + NT * i >= nreal ? 8 : 0);
#pragma unroll
                for (int j = 0; j < 8; ++j) sv[i][j] = j < mine ? 0.f : sv[i][j];
            }
        }
    };
    auto store_px = [&](char *buf) {
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
            v4u pc[3];
            split8(sv[i], pc);
#pragma unroll
            for (int q = 0; q < 3; ++q) *reinterpret_cast<v4u *>(buf + loff[i] + q * 32) = pc[q];
        }
    };

    // A: this lane's filter row, channels half*8 .. +7 of the chunk
    const int m = m0 + wm * 32 + l32;
    const unsigned aoff = m < p.M ? (unsigned)(half * 8 * T * p.M + m) * 4u : kOOB;
    auto load_a = [&](int ch, int tap, float *r) {
        const unsigned d = (unsigned)(chan0(ch) * T + tap) * (unsigned)p.M * 4u;
        const __amdgpu_buffer_rsrc_t rw =
            make_rsrc(reinterpret_cast<const char *>(p.wt) + d, wbytes - d);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            r[j] = bload_so(rw, aoff, (unsigned)(j * T) * (unsigned)p.M * 4u);
    };

    // B: this lane's output columns
    int bbase[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        int n = n0 + (wn * NF + f) * 32 + l32;
        if (n >= p.N) n = n0;
        const int b = fdiv(n, p.dohw), pos = n - b * OHW;
        const int oh = fdiv(pos, p.dow), ow = pos - oh * p.OW;
        bbase[f] = ((b * p.VH + oh - vs) * p.PW + ow) * SP_PXB + half * 16;
    }

    v16f hi[NF], lo[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < 16; ++r) hi[f][r] = lo[f][r] = 0.f;

    // every group of the workgroup runs p.cps chunks (a group past its last
    // chunk only joins the barriers)
    // The filter pipeline: in tap t the pieces of tap t multiply, the raw
    // values of tap t+1 are split and those of tap t+1+AD are loaded (the
    // fewer MFMAs a tap has, the more taps it takes to cover a load).
    constexpr int AD = 4 / NF;
    float ar[AD][8];
    v4u a[2][3];
    if (ch0 < ch1) {
        float first[8];
        load_px(ch0);
        load_a(ch0, 0, first);
#pragma unroll
        for (int t = 1; t <= AD; ++t) load_a(ch0, t, ar[t % AD]);
        store_px(stage);
        split8(first, a[0]);
    }
    __syncthreads();
    int cur = 0;
    auto compute = [&](const char *buf, int ch, bool next) {
        v4u b[2][3];
        auto load_b = [&](int step) {  // step = tap * NF + f
            const int tap = step / NF, f = step % NF;
            const char *src = buf + bbase[f] + ((tap / KS) * p.PW + tap % KS) * SP_PXB;
#pragma unroll
            for (int q = 0; q < 3; ++q) b[step & 1][q] = *reinterpret_cast<const v4u *>(src + q * 32);
        };
        load_b(0);
#pragma unroll
        for (int tap = 0; tap < T; ++tap) {
            __builtin_amdgcn_sched_barrier(0);
            const v4u *ca = a[tap & 1];
            split8(ar[(tap + 1) % AD], a[(tap + 1) & 1]);
            const int ahead = tap + 1 + AD;
            if (ahead < T) load_a(ch, ahead, ar[ahead % AD]);
            else load_a(next ? ch + 1 : ch, ahead - T, ar[ahead % AD]);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const int step = tap * NF + f;
                if (step + 1 < T * NF) load_b(step + 1);
                const v4u *c = b[step & 1];
                lo[f] = MFMA_BF(as_bf(ca[2]), as_bf(c[0]), lo[f]);
                hi[f] = MFMA_BF(as_bf(ca[0]), as_bf(c[0]), hi[f]);
                lo[f] = MFMA_BF(as_bf(ca[0]), as_bf(c[2]), lo[f]);
                lo[f] = MFMA_BF(as_bf(ca[1]), as_bf(c[1]), lo[f]);
                lo[f] = MFMA_BF(as_bf(ca[1]), as_bf(c[0]), lo[f]);
                lo[f] = MFMA_BF(as_bf(ca[0]), as_bf(c[1]), lo[f]);
            }
#pragma unroll
            for (int i = 0; i < 6 * NF; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (i % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                if (i % 3 == 0) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
        }
        // the next chunk's tap 0 and the raw values move to where it expects
        // them (the taps of a chunk are an odd number)
        static_assert(T % 2 == 1 && T % AD == 1 % AD && T > AD, "slots of the filter pipeline");
#pragma unroll
        for (int q = 0; q < 3; ++q) a[0][q] = a[1][q];
        if constexpr (AD > 1) {
            float t[AD][8];
#pragma unroll
            for (int i = 0; i < AD; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) t[i][j] = ar[(T + i) % AD][j];
#pragma unroll
            for (int i = 0; i < AD; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) ar[i][j] = t[i][j];
        }
    };
    for (int it = 0; it < p.cps; ++it) {
        const int ch = ch0 + it;
        const bool live = ch < ch1, next = ch + 1 < ch1;
        if (live) {
            const char *buf = stage + cur * bufb;
            if (next) load_px(ch + 1);
            compute(buf, ch, next);
        }
        if (p.nbuf == 1) __syncthreads();
        if (p.nbuf == 2) cur ^= 1;
        if (live && next) store_px(stage + cur * bufb);
        __syncthreads();
    }
    bool bad = false;
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            hi[f][r] += lo[f][r];
            bad |= !(fabsf(hi[f][r]) <= 3.402823466e38f);
        }
    if (__ballot(bad)) {  // this wave's tile again on the fp32 instructions
        int xo[NF], oy[NF], ox[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const int n = n0 + (wn * NF + f) * 32 + l32;
            const int b = fdiv(n, p.dohw), pos = n - b * OHW, oh = fdiv(pos, p.dow);
            oy[f] = n < p.N ? oh - p.P : p.H;  // (past the end: no row is inside)
            ox[f] = pos - oh * p.OW - p.P;
            xo[f] = b * p.C * HW + oy[f] * p.W + ox[f];
#pragma unroll
            for (int r = 0; r < 16; ++r) hi[f][r] = lo[f][r] = 0.f;
        }
        const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, xbytes), rw = make_rsrc(p.wt, wbytes);
        const int cend = min(p.C, ch1 * SP_CH);
#pragma unroll 1
        for (int c0 = ch0 * SP_CH; c0 < cend; c0 += 2) {  // lane half h: channel c0 + h
            const int c = c0 + half;
            // a chunk's sums stand by themselves: one chain over all channels
            // had up to twice the error of the fp32 kernels' K parts
            if (c0 % SP_CH == 0) {
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    hi[f] += lo[f];
#pragma unroll
                    for (int r = 0; r < 16; ++r) lo[f][r] = 0.f;
                }
            }
#pragma unroll 1
            for (int ki = 0; ki < KS; ++ki) {
                float av[KS], bv[NF][KS];
#pragma unroll
                for (int kj = 0; kj < KS; ++kj) {
                    av[kj] = bload(rw, boff((c < cend) & (m < p.M),
                                            (c * T + ki * KS + kj) * p.M + m));
#pragma unroll
                    for (int f = 0; f < NF; ++f)
                        bv[f][kj] = bload(rx, boff((c < cend) & ((unsigned)(oy[f] + ki) < (unsigned)p.H) &
                                                       ((unsigned)(ox[f] + kj) < (unsigned)p.W),
                                                   xo[f] + c * HW + ki * p.W + kj));
                }
#pragma unroll
                for (int kj = 0; kj < KS; ++kj)
#pragma unroll
                    for (int f = 0; f < NF; ++f)
                        lo[f] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[kj], bv[f][kj], lo[f], 0, 0, 0);
            }
        }
#pragma unroll
        for (int f = 0; f < NF; ++f) hi[f] += lo[f];
    } else {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r) hi[f][r] *= kSumDown;
    }
    // each group hands the other the half of the fragments that one stores
    if constexpr (KG == 2) {
        static_assert(NF % 2 == 0 || KG == 1, "the groups exchange half of the fragments each");
        float4 *xs = reinterpret_cast<float4 *>(smem);
        constexpr int HF = NF / 2;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if (f / HF == grp) continue;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                xs[(f * 4 + r4) * NT + tid] = make_float4(hi[f][4 * r4], hi[f][4 * r4 + 1],
                                                          hi[f][4 * r4 + 2], hi[f][4 * r4 + 3]);
        }
        __syncthreads();
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if (f / HF != grp) continue;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const float4 o = xs[(f * 4 + r4) * NT + tid];
                hi[f][4 * r4] += o.x;
                hi[f][4 * r4 + 1] += o.y;
                hi[f][4 * r4 + 2] += o.z;
                hi[f][4 * r4 + 3] += o.w;
            }
        }
    }
    // D layout: lane l, register r holds row 8*(r/4) + 4*(l/32) + r%4,
    // column l%32
    const int mb = m0 + wm * 32 + 4 * half;
    const bool full = m0 + 32 * WM <= p.M;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        if (KG == 2 && f / (NF / 2 > 0 ? NF / 2 : 1) != grp) continue;
        const int n = n0 + (wn * NF + f) * 32 + l32;
        if (n >= p.N) continue;
        float *base;
        int stride;
        if (p.splits > 1) {
            base = p.part + ((size_t)z * p.M + mb) * p.N + n;
            stride = p.N;
        } else {
            const int b = fdiv(n, p.dohw), pos = n - b * OHW;
            base = p.y + ((size_t)b * p.M + mb) * OHW + pos;
            stride = OHW;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int dm = 8 * (r >> 2) + (r & 3);
            if (full || mb + dm < p.M) {
                float v = hi[f][r];
                if constexpr (EPI) v = p.e.apply(v, mb + dm);
                base[(size_t)dm * stride] = v;
            }
        }
    }
}

// The most patch pixels (padding included) and input pixels that a
// 128-position tile can need
static void split_patch(const ConvGeom &g, long long &npx, long long &nreal)
{
    const int ohw = g.OH * g.OW, pw = g.OW + g.KS - 1, vh = g.OH + g.KS - 1;
    long long imgs, rows;  // images and output rows a tile touches
    if (ohw % SP_BN == 0) imgs = 1;
    else if (SP_BN % ohw == 0) imgs = SP_BN / ohw;
    else imgs = (SP_BN - 2) / ohw + 2;
    if (g.OW % SP_BN == 0) rows = 1;
    else if (SP_BN % g.OW == 0 && ohw % SP_BN == 0) rows = SP_BN / g.OW;
    else if (SP_BN % ohw == 0) rows = imgs * g.OH;
    else rows = (SP_BN - 2) / g.OW + 2;
    if (imgs > g.B) imgs = g.B;
    if (rows > (long long)g.B * g.OH) rows = (long long)g.B * g.OH;
    const long long vrows = rows + imgs * (g.KS - 1);
    npx = (vrows < (long long)g.B * vh ? vrows : (long long)g.B * vh) * pw;
    // each image's rows r read at most r + KS-1-P input rows up to the
    // image's edge, and a tile inside one image at most r + KS-1
    const long long edge = imgs * (g.KS - 1 - g.P);
    long long real = rows + (edge > g.KS - 1 ? edge : g.KS - 1);
    if (SP_BN % ohw == 0 || real > imgs * g.H) real = imgs * g.H;
    nreal = real * g.W;
}

// 72 steps, 128 -> 128 @ 32x32: 2.0e-7, after a relu 1.5e-7.  (128 -> 96 5x5 at
// 20x56, batch 8, in one chain of 200 steps was at 3.4e-7, the fp32 kernel with
// 13 parts at 2.7e-7.)
constexpr StepError kStepError = {1.8, 1.25};

// Up to 32 filters a workgroup has little work for its loads, and small grids
// of them can be slower than the fp32 kernel's: 144 -> 16 5x5 at 45x32, one
// image, 21.6 us, 14.4 on fp32.  Both times (us) by models fitted to 4700 such
// layers, within 6% on eight of ten (one set of constants for 3x3, one for
// 5x5): a step of a chunk (or k-tile) with one workgroup on every CU and with
// more, the partial sums in MB, workgroups in thousands.
struct NarrowTime {
    double fix, one, more, split, mb, wgs;
};
constexpr NarrowTime kNarrowPieces[2] = {{6.1, 2.4, 3.9, 2.9, 0.19, 3.2}, {5.9, 2.1, 3.3, 2.5, 0.25, 3.1}};
constexpr NarrowTime kNarrowFp32[2] = {{4.9, 0.59, 0.28, 2.9, 0.20, 2.3}, {4.7, 0.96, 0.34, 1.4, 0.29, 3.9}};

static bool narrow_pays(const ConvGeom &g, const SplitFwdPlan &pl, const Fp32Fwd &fp32)
{
    const double mn = (double)g.F * g.B * g.OH * g.OW * 4e-6, taps = g.KS * g.KS / 9.0;
    const int nchunk = (g.C + SP_CH - 1) / SP_CH, cps = (nchunk + pl.splits - 1) / pl.splits;
    const long long wgs = ((long long)g.B * g.OH * g.OW + SP_BN - 1) / SP_BN * pl.splits;
    const NarrowTime &p = kNarrowPieces[g.KS == 5], &f = kNarrowFp32[g.KS == 5];
    const long long full = wgs / 512, rest = wgs % 512;
    double tp = p.fix + cps * taps * (full * p.more + (rest > 256 ? p.more : rest ? p.one : 0.0)) +
                p.wgs * wgs / 1000;
    if (pl.splits > 1) tp += p.split + p.mb * (2 * pl.splits + 1) * mn;
    const double wf = (double)fp32.tiles * fp32.parts;
    double tf = f.fix + fp32.ktiles * (f.one + f.more * (wf > 256 ? wf / 256 - 1 : 0.0)) +
                f.wgs * wf / 1000;
    if (fp32.slices > 1) tf += f.split + f.mb * (2 * fp32.slices + 1) * mn;
    return tp < tf;
}

SplitFwdPlan split_fwd_plan(const ConvGeom &g, bool kg_ok, const Fp32Fwd &fp32, int room)
{
    SplitFwdPlan pl{};
    pl.ok = false;
    if (g.S != 1 || !(g.KS == 3 || g.KS == 5) || g.P > g.KS - 1 || g.C < SP_CH) return pl;
    // chunks that are mostly repeated channels (17-22, 33) lose to the fp32
    // kernel (18 -> 16 @ 39x39, batch 5: 9.9 against 11.0 us)
    if (g.C < 0.7 * SP_CH * ((g.C + SP_CH - 1) / SP_CH)) return pl;
    if ((long long)g.B * (g.OH + g.KS) >= (1ll << 30)) return pl;
    const int M = g.F, N = g.B * g.OH * g.OW;
    long long npx, nreal;
    split_patch(g, npx, nreal);
    if (npx * SP_PXB > 150 * 1024) return pl;
    pl.npx = (int)npx;
    const int nchunk = (g.C + SP_CH - 1) / SP_CH, nt = (N + SP_BN - 1) / SP_BN;
    const int wide = M <= 32 ? 1 : (M <= 64 ? 2 : (M <= 96 ? 3 : 4));
    const long long big = (long long)((M + 127) / 128) * nt;  // 128 x 128 tiles
    // Waves along M and K parts: the modelled time of the rounds of workgroups,
    // two per CU (or one with two K groups), plus the split-K reduction.  us per
    // 16-channel chunk of a 3x3 filter with two workgroups on every CU and with
    // one, by waves along M, fitted to a sweep of 30 layers that ran each height
    // in turn (one wave's 32 rows: every wave loads the filter rows again).
    // Against fixed prices of 11 / 6.2 / 3.6 us for 3-4 / 2 / 1 waves: 256 -> 96
    // 5x5 at 27x27, batch 128: 692 -> 555 us; 128 -> 128 at 32x32, batch 40:
    // 88 -> 72.  Small grids take no more slices than the fp32 plan.
    static const double kPaired[5] = {0, 4.1, 5.8, 8.0, 10.6};
    static const double kSingle[5] = {0, 2.5, 3.5, 5.2, 7.0};
    double best = -1;
    for (int wm = wide; wm >= 1; wm = wm == 4 ? 2 : wm - 1) {
        const int wn = wm == 1 ? 4 : (wm == 2 ? 2 : 1), thr = 64 * wm * wn;
        const long long tpt = (2 * nreal + thr - 1) / thr;
        const long long tiles = (long long)((M + 32 * wm - 1) / (32 * wm)) * nt;
        if (tpt > 4 || tiles > 0x7fffffffLL) continue;
        const double taps = g.KS * g.KS / 9.0;
        const double paired = kPaired[wm] * taps, single = kSingle[wm] * taps;
        for (int kg = 1; kg <= (kg_ok && wm == 4 && tpt <= 3 ? 2 : 1); ++kg)
            for (const int s : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 24, 32}) {
                if (s * kg > nchunk || (s > 1 && tiles * s > 2048)) break;
                const int cps = (nchunk + s * kg - 1) / (s * kg);
                const int splits = (nchunk + cps * kg - 1) / (cps * kg);
                if (!no_more_error(kStepError, cps * g.KS * g.KS, splits * kg,
                                   (double)g.C * g.KS * g.KS / fp32.parts, fp32.parts))
                    continue;
                if (splits > 1 && (splits > room || (splits > fp32.slices && big < 128))) continue;
                const long long wgs = tiles * splits;
                const long long full = wgs >> (kg == 2 ? 8 : 9), rest = wgs & (kg == 2 ? 255 : 511);
                double t = full * cps * paired;
                if (rest) t += cps * (rest > 256 || kg == 2 ? paired : single);
                if (splits > 1) t += 5.0 + (2.0 * splits + 1) * M * (double)N * 4 / 5e6;
                if (best < 0 || t < best * 0.97) {
                    best = t;
                    pl.wm = wm;
                    pl.wn = wn;
                    pl.kg = kg;
                    pl.splits = splits;
                    pl.tpt = tpt < 2 ? 2 : (int)tpt;
                }
            }
    }
    if (best < 0) return pl;
    const int one = (pl.npx + 1) * SP_PXB;
    // two workgroups (or two K groups) share a CU's 160 KB
    pl.nbuf = 2 * one <= 80 * 1024 ? 2 : 1;
    pl.ok = pl.kg * pl.nbuf * one <= SP_LDS && (M > 32 || narrow_pays(g, pl, fp32));
    return pl;
}

template <int WM, int WN, int KG, int KS, int TPT>
static int split_go(const SplitFwd &p, const SplitFwdPlan &pl, hipStream_t st)
{
    size_t lds = (size_t)KG * pl.nbuf * (pl.npx + 1) * SP_PXB;
    if (KG == 2) {
        const size_t xch = (size_t)4 * 4 * 64 * WM * WN * sizeof(float4);
        if (lds < xch) lds = xch;
    }
    const bool epi = p.e.active() && p.splits == 1;
    auto kern = epi ? &k_conv_split<WM, WN, KG, KS, TPT, true>
                    : &k_conv_split<WM, WN, KG, KS, TPT, false>;
    if (lds > 64 * 1024) {
        // the CU's LDS, not this launch's size: the limit is the kernel's for
        // the whole process, and another thread may launch the same kernel
        // with a smaller patch between these two calls
        const int rc = check(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 SP_LDS));
        if (rc) return rc;
    }
    hipLaunchKernelGGL(kern, dim3(p.tiles, p.splits), dim3(64 * WM * WN * KG), lds, st, p);
    return check_launch();
}

template <int KS, int TPT>
static int split_ks(const SplitFwd &p, const SplitFwdPlan &pl, hipStream_t st)
{
    if (pl.wm == 1) return split_go<1, 4, 1, KS, TPT>(p, pl, st);
    if (pl.wm == 2) return split_go<2, 2, 1, KS, TPT>(p, pl, st);
    if (pl.wm == 3) return split_go<3, 1, 1, KS, TPT>(p, pl, st);
    if constexpr (TPT <= 3)
        if (pl.kg == 2) return split_go<4, 1, 2, KS, TPT>(p, pl, st);
    return split_go<4, 1, 1, KS, TPT>(p, pl, st);
}

template <int KS>
static int split_tpt(const SplitFwd &p, const SplitFwdPlan &pl, hipStream_t st)
{
    if (pl.tpt == 2) return split_ks<KS, 2>(p, pl, st);
    if (pl.tpt == 3) return split_ks<KS, 3>(p, pl, st);
    return split_ks<KS, 4>(p, pl, st);
}

int split_fwd_launch(const ConvGeom &g, const SplitFwdPlan &pl, const float *x, const float *wt,
                     float *y, float *part, const Epi &e, hipStream_t st)
{
    SplitFwd p{};
    p.x = x; p.wt = wt; p.y = y; p.part = part;
    p.B = g.B; p.C = g.C; p.H = g.H; p.W = g.W; p.M = g.F;
    p.P = g.P; p.OH = g.OH; p.OW = g.OW;
    p.N = g.B * g.OH * g.OW;
    p.VH = g.OH + g.KS - 1;
    p.PW = g.OW + g.KS - 1;
    p.nchunk = (g.C + SP_CH - 1) / SP_CH;
    p.cps = (p.nchunk + pl.splits * pl.kg - 1) / (pl.splits * pl.kg);
    p.splits = pl.splits;
    p.nbuf = pl.nbuf;
    p.npx = pl.npx;
    p.mt = (g.F + 32 * pl.wm - 1) / (32 * pl.wm);
    const long long tiles = (long long)p.mt * ((p.N + SP_BN - 1) / SP_BN);
    if (tiles > 0x7fffffffLL) return ACH_EINVAL;
    p.tiles = (int)tiles;
    p.dohw = make_fastdiv((unsigned)(g.OH * g.OW));
    p.dow = make_fastdiv((unsigned)g.OW);
    p.dh = make_fastdiv((unsigned)g.H);
    p.dw = make_fastdiv((unsigned)g.W);
    p.e = e;
    if (g.KS == 3) return split_tpt<3>(p, pl, st);
    return split_tpt<5>(p, pl, st);
}

}  // namespace ach
