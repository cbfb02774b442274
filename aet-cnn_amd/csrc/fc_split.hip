// Fully connected layers' GEMMs on the bf16 matrix cores, every float as three
// exact bf16 pieces (the arithmetic and the treatment of non-finite values of
// conv_split.hip).
//
// One kernel for the three passes: 128 x 128 tiles (64 x 128 for up to 64
// rows), rows the batch (forward, input gradient) or the filters (weight
// gradient), columns the features.  A chunk of 32 k of both operands is loaded
// a chunk ahead (a lane 8 consecutive k of one row: two 16-byte loads from a
// row-major operand, eight coalesced dwords from a k-major one), split and
// staged in LDS as [row][3 pieces][32 k], 208 bytes a row, which keeps both
// sides' 16-byte accesses free of bank conflicts.
//
// Bound: memory in the weight gradient (reads and writes dw: 302 MB of the
// 9216 x 4096 layer), the split's VALU work and the latency of one chunk at
// a time elsewhere.  Batch 128, fp32 kernels before -> now: 9216 -> 4096
// forward 105 -> 65 us, input gradient 161 -> 70, weight gradient 128 -> 124;
// 4096 -> 4096 55 -> 37, 52 -> 39, 86 -> 55; error against 64 bits 0.33-0.43 of
// theirs.  Up to 32 rows a tile is mostly padding and the fp32 kernels stay;
// so do they for weight gradients of at most 64 images (48, 4096 -> 4096: 38
// against 47 us) or fewer than 512 tiles.
#include "fc_split.hpp"
#include "pieces.hpp"

namespace ach {

constexpr int FP_K = 32;       // k per chunk
constexpr int FP_ROWB = 208;   // LDS bytes per row

struct FcSplit {
    const float *a, *b;
    float *y, *part;
    int R, N, K, cps, slices, nt;
    Epi e;
    Sgd sg;
};

// AK / BKM: the operand is k-major.  MODE 0: forward / input gradient store;
// 1: with the epilogue; 2: weight gradient (y += the sums, then SGD)
template <int MT, int WM, bool AK, bool BKM, int MODE>
__global__ void __launch_bounds__(256, 2) k_fc_split(FcSplit p)
{
    constexpr int WN = 4 / WM, NT = 4 / WN, MR = 32 * MT * WM;
    constexpr int ATASK = MR * 4 / 256, BTASK = 2;
    __shared__ __align__(16) char smem[(MR + 128) * FP_ROWB];
    char *const sa = smem, *const sb = smem + MR * FP_ROWB;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM, half = lane >> 5, l32 = lane & 31;
    int id = blockIdx.x;
    {
        const int G = gridDim.x, g8 = G >> 3, r8 = G & 7, xcd = id & 7, k = id >> 3;
        id = xcd * g8 + min(xcd, r8) + k;
    }
    const int z = blockIdx.y;
    const int n0 = (id % p.nt) * 128, m0 = (id / p.nt) * MR;
    const int k0 = z * p.cps * FP_K, k1 = min(p.K, k0 + p.cps * FP_K);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.a, (unsigned)((size_t)p.R * p.K * 4));
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(p.b, (unsigned)((size_t)p.N * p.K * 4));

    // task t of an operand: row and segment of 8 k.  Row-major: the four
    // segments of a row on adjacent lanes; k-major: adjacent lanes on
    // adjacent rows
    auto load = [&](__amdgpu_buffer_rsrc_t rs, bool km, int t, int rows, int base, int total, int kc,
                    float *v) {
        const int q = tid + 256 * t;
        const int row = base + (km ? q % rows : q >> 2), k = kc + (km ? q / rows : q & 3) * 8;
        if (km) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                v[j] = bload(rs, boff((row < total) & (k + j < k1), (k + j) * total + row));
        } else if ((p.K & 7) == 0) {  // k1 and k are multiples of 8
            const int o = boff((row < total) & (k < k1), row * p.K + k);
            const float4 x = bload4_so(rs, o, 0), y = bload4_so(rs, o, 16);
            v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
            v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                v[j] = bload(rs, boff((row < total) & (k + j < k1), row * p.K + k + j));
        }
    };
    auto store = [&](char *s, bool km, int t, int rows, const float *v) {
        const int q = tid + 256 * t;
        const int row = km ? q % rows : q >> 2, seg = km ? q / rows : q & 3;
        v4u pc[3];
        split8(v, pc);
        char *dst = s + row * FP_ROWB + seg * 16;
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<v4u *>(dst + i * 64) = pc[i];
    };
    float va[ATASK][8], vb[BTASK][8];
    auto load_all = [&](int kc) {
#pragma unroll
        for (int t = 0; t < ATASK; ++t) load(ra, AK, t, MR, m0, p.R, kc, va[t]);
#pragma unroll
        for (int t = 0; t < BTASK; ++t) load(rb, BKM, t, 128, n0, p.N, kc, vb[t]);
    };

    v16f hi[MT][NT], lo[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) hi[i][j][e] = lo[i][j][e] = 0.f;

    load_all(k0);
    for (int kc = k0; kc < k1; kc += FP_K) {
#pragma unroll
        for (int t = 0; t < ATASK; ++t) store(sa, AK, t, MR, va[t]);
#pragma unroll
        for (int t = 0; t < BTASK; ++t) store(sb, BKM, t, 128, vb[t]);
        __syncthreads();
        load_all(kc + FP_K);  // past k1: zeros
#pragma unroll
        for (int s = 0; s < FP_K / 16; ++s) {
            v4u a[MT][3];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    a[i][q] = *reinterpret_cast<const v4u *>(
                        sa + ((wm * MT + i) * 32 + l32) * FP_ROWB + q * 64 + (s * 2 + half) * 16);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                v4u b[3];
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    b[q] = *reinterpret_cast<const v4u *>(
                        sb + ((wn * NT + j) * 32 + l32) * FP_ROWB + q * 64 + (s * 2 + half) * 16);
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    lo[i][j] = MFMA_BF(as_bf(a[i][2]), as_bf(b[0]), lo[i][j]);
                    hi[i][j] = MFMA_BF(as_bf(a[i][0]), as_bf(b[0]), hi[i][j]);
                    lo[i][j] = MFMA_BF(as_bf(a[i][0]), as_bf(b[2]), lo[i][j]);
                    lo[i][j] = MFMA_BF(as_bf(a[i][1]), as_bf(b[1]), lo[i][j]);
                    lo[i][j] = MFMA_BF(as_bf(a[i][1]), as_bf(b[0]), lo[i][j]);
                    lo[i][j] = MFMA_BF(as_bf(a[i][0]), as_bf(b[1]), lo[i][j]);
                }
            }
        }
        __syncthreads();
    }
    // the weight gradient's prior values, all loads in flight at once
    float old[MODE == 2 ? MT : 1][NT][16];
    auto load_old = [&](auto each) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int r = m0 + (wm * MT + i) * 32 + 4 * half, c = n0 + (wn * NT + j) * 32 + l32;
                const float *base = p.y + (size_t)r * p.N + c;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int dr = 8 * (e >> 2) + (e & 3);
                    each(i, j, e);
                    old[i][j][e] = c < p.N && r + dr < p.R ? base[(size_t)dr * p.N] : 0.f;
                }
            }
    };
    if constexpr (MODE == 2)
        load_old([&](int i, int j, int e) { hi[i][j][e] += lo[i][j][e]; });
    bool bad = false;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                if constexpr (MODE != 2) hi[i][j][e] += lo[i][j][e];
                bad |= !(fabsf(hi[i][j][e]) <= 3.402823466e38f);
            }
    float down = kSumDown;
    if (__ballot(bad)) {  // this wave's tiles again on the fp32 instructions
        down = 1.f;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) hi[i][j][e] = lo[i][j][e] = 0.f;
        auto at = [&](bool km, int row, int total, int k) {
            return boff((row < total) & (k < k1), km ? k * total + row : row * p.K + k);
        };
        // (a chunk's sums stand by themselves: one chain had up to 1.4 times
        // the error of the fp32 kernels' K parts)
        constexpr int U = 4;
#pragma unroll 1
        for (int kc = k0; kc < k1; kc += 2 * U) {  // lane half h: k = kc + 2u + h
            if (((kc - k0) & (FP_K - 1)) == 0) {
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) {
                        hi[i][j] += lo[i][j];
#pragma unroll
                        for (int e = 0; e < 16; ++e) lo[i][j][e] = 0.f;
                    }
            }
            float av[U][MT], bv[U][NT];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = kc + 2 * u + half;
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    av[u][i] = bload(ra, at(AK, m0 + (wm * MT + i) * 32 + l32, p.R, k));
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    bv[u][j] = bload(rb, at(BKM, n0 + (wn * NT + j) * 32 + l32, p.N, k));
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        lo[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[u][i], bv[u][j], lo[i][j],
                                                                        0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) hi[i][j] += lo[i][j];
        // (read again: kept over the recomputation they would not fit)
        if constexpr (MODE == 2) load_old([](int, int, int) {});
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int r = m0 + (wm * MT + i) * 32 + 4 * half, c = n0 + (wn * NT + j) * 32 + l32;
            if (c >= p.N) continue;
            if constexpr (MODE == 2) {
                float *base = p.y + (size_t)r * p.N + c, wv[16];
                float *wb = p.sg.w ? p.sg.w + (size_t)r * p.N + c : nullptr;
                if (wb) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int dr = 8 * (e >> 2) + (e & 3);
                        wv[e] = r + dr < p.R ? wb[(size_t)dr * p.N] : 0.f;
                    }
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int dr = 8 * (e >> 2) + (e & 3);
                    if (r + dr >= p.R) continue;
                    float u = old[i][j][e] + hi[i][j][e] * down;
                    if (wb) {
                        sgd_step(wv[e], u, p.sg.dc, p.sg.lc, p.sg.mom);
                        wb[(size_t)dr * p.N] = wv[e];
                    }
                    base[(size_t)dr * p.N] = u;
                }
            } else {
                float *base = p.slices > 1 ? p.part + ((size_t)z * p.R + r) * p.N + c
                                           : p.y + (size_t)r * p.N + c;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int dr = 8 * (e >> 2) + (e & 3);
                    float v = hi[i][j][e] * down;
                    if constexpr (MODE == 1) v = p.e.apply(v, c);
                    if (r + dr < p.R) base[(size_t)dr * p.N] = v;
                }
            }
        }
}

int fc_split_slices(int batch, int features, int K, int room)
{
    if (batch <= 32 || features < 128 || K < 128) return 0;
    const int mr = batch <= 64 ? 64 : 128;
    const int tiles = ((features + 127) / 128) * ((batch + mr - 1) / mr);
    const int chunks = (K + FP_K - 1) / FP_K;
    int s = tiles < 512 ? 512 / tiles : 1;
    const int least = tiles < 32 ? 2 : 4;  // chunks per slice
    if (s > chunks / least) s = chunks / least;
    if (s > 32) s = 32;
    if (s > room) s = room;
    if (s < 1) s = 1;
    const int cps = (chunks + s - 1) / s;
    return (chunks + cps - 1) / cps;
}

template <bool AK, bool BKM, int MODE>
static int fc_go(const FcSplit &p, hipStream_t st)
{
    if (p.R <= 64) {
        hipLaunchKernelGGL((k_fc_split<2, 1, AK, BKM, MODE>), dim3(p.nt * ((p.R + 63) / 64), p.slices),
                           dim3(256), 0, st, p);
    } else {
        hipLaunchKernelGGL((k_fc_split<2, 2, AK, BKM, MODE>),
                           dim3(p.nt * ((p.R + 127) / 128), p.slices), dim3(256), 0, st, p);
    }
    return check_launch();
}

int fc_split_launch(const FcOperand &a, const FcOperand &b, int K, int slices, float *y,
                    float *part, const Epi &e, hipStream_t st)
{
    FcSplit p{};
    p.a = a.p; p.b = b.p; p.y = y; p.part = part;
    p.R = a.rows; p.N = b.rows; p.K = K;
    p.cps = ((K + FP_K - 1) / FP_K + slices - 1) / slices;
    p.slices = slices;
    p.nt = (p.N + 127) / 128;
    p.e = e;
    if (a.kmajor) return ACH_EINVAL;
    if (e.active() && slices == 1)
        return b.kmajor ? fc_go<false, true, 1>(p, st) : fc_go<false, false, 1>(p, st);
    return b.kmajor ? fc_go<false, true, 0>(p, st) : fc_go<false, false, 0>(p, st);
}

bool fc_split_wgrad(int F, int C, int batch)
{
    return batch > 64 && (long long)((F + 127) / 128) * ((C + 127) / 128) >= 512;
}

int fc_split_wgrad_launch(int F, int C, int batch, const float *dy, const float *x, float *dw,
                          const Sgd &sg, hipStream_t st)
{
    FcSplit p{};
    p.a = dy; p.b = x; p.y = dw;
    p.R = F; p.N = C; p.K = batch;
    p.cps = (batch + FP_K - 1) / FP_K;
    p.slices = 1;
    p.nt = (C + 127) / 128;
    p.sg = sg;
    hipLaunchKernelGGL((k_fc_split<2, 2, true, true, 2>), dim3(p.nt * ((F + 127) / 128)), dim3(256), 0,
                       st, p);
    return check_launch();
}

}  // namespace ach
