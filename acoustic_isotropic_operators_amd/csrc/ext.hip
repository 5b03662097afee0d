// ext.hip -- secondary sources and imaging of the offset extension with four
// z-points per lane.
//
// What bounds the secondary sources: the latency of one sample's pieces per barrier, with two
// workgroups of 8 waves per CU (230 vector instructions per 256 points and
// sample, 168 of them the products and sums; no LDS conflicts).  All offsets
// are computed without a test, those beyond 2 hExt on zeros: with a branch per
// offset every LDS read was waited for.  64 x 32 tiles stage 2.25 times their
// points, the one-point kernels' 64 x 16 ones 3.5 times.  Not built for more
// than 21 offsets: the model values of 41 would take 164 registers and leave
// one workgroup per CU; that form was not measured.
// Extended forward, 6 shots of 500 x 1200, 21 offsets, 300 samples: 27.2 ms,
// one point per lane 30.3; tomographic adjoint, 6 shots of 300 x 700: 33.1 ms,
// 37.1.  Up to 11 offsets both take the same time, and the one-point kernels
// stay.
#include <hip/hip_runtime.h>

#include "wide.hpp"

namespace aiso {

namespace {

constexpr int kTZ = 64, kTX = 32, kQ = kTZ / 4, kThreads = kQ * kTX;
constexpr int kShots = 2;   // shots per workgroup, which share its model values

// For the nk samples of each shot, into ss[0] + ssOff[k], over the offsets h =
// -hExt .. hExt in order:
//   ss_k[x] = v2dt2[x] * sum m[h][x-h] * W_k[x-2h]              (k_ext_ss_tile)
//   TOMO: ss_k[x] = sum (m[h][x+h] * W_k[x+2h]) * v2dt2[x+2h]    (k_tomo_adj_ss_tile)
// Each thread owns four rows of one column and keeps its model values in
// registers; W passes through LDS in 16-byte pieces, the next sample's loaded
// while the current one is computed, into the other half: one barrier per
// sample.  Offsets that leave the interior have a model value of zero.
template <int HX, bool TOMO>
__global__ __launch_bounds__(kThreads) void k_offset_ss(ExtBatchArgs a, int nshots, int nbx, int nbz, int nby)
{
    constexpr int NE = 2 * HX + 1, LW = kTX + 4 * HX, SZ = LW * kTZ, KU = (LW * kQ + kThreads - 1) / kThreads;
    __shared__ __attribute__((aligned(16))) float lds[(TOMO ? 3 : 2) * SZ];
    const int l = xcd_logical(blockIdx.x, gridDim.x);
    if (l >= nbx * nbz * nby) return;                                           // padding blocks (block-uniform)
    const int bx = l % nbx, bz = l / nbx % nbz, by = l / nbx / nbz, t = threadIdx.x;
    const int hExt = a.hExt, ne = 2 * hExt + 1, lw = kTX + 4 * hExt, nzi = a.nz - 2 * FAT;
    const int z0 = bz * kTZ, x0 = FAT + bx * kTX;                               // interior row, grid column
    const long nzx = (long)a.nz * a.nx;
    // Offset e takes LDS column c + 2e (TOMO) or c + 4 HX - 2e, whatever hExt
    // is: column j is grid column x0 - 2 hExt + j (TOMO) or x0 + 2 hExt - 4 HX
    // + j.  Columns outside the interior and those that only offsets beyond
    // 2 hExt take are zero.
    unsigned off[KU];
    bool in[KU];
    f4 pre[KU];
#pragma unroll
    for (int k = 0; k < KU; ++k) {
        const int u = t + k * kThreads, j = u / kQ - (TOMO ? 0 : 4 * (HX - hExt)), q = u % kQ, gx = x0 - 2 * hExt + j;
        in[k] = j >= 0 && j < lw && gx >= FAT && gx < a.nx - FAT && z0 + 4 * q < nzi;
        off[k] = in[k] ? 4u * (unsigned)(gx * a.nz + FAT + z0 + 4 * q) : 0u;
        pre[k] = (f4)0.f;
    }
    auto fetch = [&](cgf* w) {
#pragma unroll
        for (int k = 0; k < KU; ++k)
            if (in[k]) pre[k] = ld4(w, off[k]);
    };
    auto store = [&](float* to) {
#pragma unroll
        for (int k = 0; k < KU; ++k)
            if (t + k * kThreads < LW * kQ) *(f4a*)&to[4 * (t + k * kThreads)] = pre[k];
    };
    const int sh0 = by * kShots, nsh = imin(kShots, nshots - sh0);
    if constexpr (TOMO) {
        fetch(G(a.v2dt2));
        store(lds + 2 * SZ);
    }
    static_assert(kShots == 2, "the bases of two shots, read before the first store");
    cgf* W0 = G(a.slots[sh0].W);
    cgf* W1 = G(a.slots[sh0 + nsh - 1].W);
    gf* S0 = G(a.slots[sh0].ss[0]);
    gf* S1 = G(a.slots[sh0 + nsh - 1].ss[0]);
    fetch(W0 + a.wOff[0]);

    const int zq = t % kQ, c = t / kQ, x = x0 + c;
    const bool ok = z0 + 4 * zq < nzi && x < a.nx - FAT;
    const unsigned o = 4u * (unsigned)(x * a.nz + FAT + z0 + 4 * zq);
    const int lo = TOMO ? max(-hExt, FAT + hExt - x) : max(-hExt, x + 1 + FAT + hExt - a.nx);
    const int hi = TOMO ? imin(a.nx - 1 - FAT - x - hExt, hExt) : imin(x - hExt - FAT, hExt);
    f4 mv[NE], vs = (f4)0.f;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        const int h = e - hExt;
        mv[e] = (f4)0.f;
        if (ok && e < ne && h >= lo && h <= hi)
            mv[e] = ld4(G(a.mext) + nzx * e + (long)(TOMO ? h : -h) * a.nz, o);
    }
    if (!TOMO && ok) vs = ld4(G(a.v2dt2), o);
    store(lds);
    __syncthreads();
    const int j0 = (TOMO ? c : c + 4 * HX) * kTZ + 4 * zq;
    int b = 0;
    for (int q = 0; q < nsh; ++q) {
        cgf* W = q ? W1 : W0;
        gf* ss = q ? S1 : S0;
        for (int k = 0; k < a.nk; ++k) {
            const bool more = k + 1 < a.nk || q + 1 < nsh;
            if (more) fetch(k + 1 < a.nk ? W + a.wOff[k + 1] : W1 + a.wOff[0]);
            const float* w = &lds[b * SZ + j0];
            const float* v = &lds[2 * SZ + j0];
            f4 acc = (f4)0.f;
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                if constexpr (TOMO) acc += (mv[e] * *(const f4a*)(w + 2 * e * kTZ)) * *(const f4a*)(v + 2 * e * kTZ);
                else acc += mv[e] * *(const f4a*)(w - 2 * e * kTZ);
            }
            if (ok) st4(ss + a.ssOff[k], o, TOMO ? acc : acc * vs);
            if (more) store(lds + (b ^ 1) * SZ);
            __syncthreads();
            b ^= 1;
        }
    }
}

// img[e][x] += (ss_k[x+h] * v2dt2[x+h]) * W_k[x-h], h = e - hExt, for x in
// [FAT+hExt, nx-FAT-hExt) and the nk samples in order (k_ext_img_tile).  A
// workgroup images every offset of a 64 x 28 tile: three groups of four waves,
// each thread NG offsets at four rows of two columns, kept in registers over the
// batch.  Every thread stages one piece of each field per sample; the next two
// samples' are loaded while two are computed, into the other half of LDS: one
// barrier per two samples.
//
// What bounds it: memory latency at one workgroup per CU.  k_ext_img_tile stages
// a 64 x 16 tile for each of three offset groups and spends 172 vector
// instructions per point and sample, four times its products.  Adjoint of 10
// shots of 400 x 1000, 21 offsets, 400 samples: 38.9 ms (43.5 with 16 samples
// per launch), k_ext_img_tile 46.8.  With three columns per thread, 64 x 48
// tiles and one sample per barrier 63 registers spilled and it took 49.7 ms.
constexpr int kImgTX = 28, kImgCX = 2, kImgGroups = 3, kImgThreads = 256 * kImgGroups;

template <int HX, int NG>
__global__ __launch_bounds__(kImgThreads) void k_offset_img(TimeBatchArgs a, int nbx, int nbz, int nshots)
{
    constexpr int LW = kImgTX + 2 * HX, SZ = LW * kTZ;
    static_assert(NG * kImgGroups >= 2 * HX + 1 && LW * kQ <= kImgThreads, "offsets of the groups, pieces of the threads");
    __shared__ __attribute__((aligned(16))) float lds[8 * SZ];                  // [half][sample][R, W]
    const int l = xcd_logical(blockIdx.x, gridDim.x);
    if (l >= nbx * nbz * nshots) return;                                        // padding blocks (block-uniform)
    const int bx = l % nbx, bz = l / nbx % nbz, shot = l / nbx / nbz;
    const int hExt = a.hExt, ne = 2 * hExt + 1, lw = kImgTX + 2 * hExt, nzi = a.nz - 2 * FAT, t = threadIdx.x;
    const int z0 = bz * kTZ, x0 = FAT + hExt + bx * kImgTX, xEnd = a.nx - FAT - hExt;   // interior row, grid column
    const long nzx = (long)a.nz * a.nx;
    const ShotSlot& S = a.slots[shot];
    cgf* ssB = G(S.ss[0]);
    cgf* WB = G(S.W);
    gf* img = G(S.img);

    // Staged column j is grid column x0 - hExt + j.
    const int gx = x0 - hExt + t / kQ;
    const bool in = t / kQ < lw && gx < a.nx && z0 + 4 * (t % kQ) < nzi;
    const unsigned off = in ? 4u * (unsigned)(gx * a.nz + FAT + z0 + 4 * (t % kQ)) : 0u;
    f4 vv = (f4)0.f, pr[2], pw[2];
    pr[0] = pr[1] = pw[0] = pw[1] = (f4)0.f;
    if (in) vv = ld4(G(a.v2dt2), off);
    auto fetch = [&](int s) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            if (in && s + j < a.nk) {
                pr[j] = ld4(ssB + a.ssOff[s + j], off);
                pw[j] = ld4(WB + a.wOff[s + j], off);
            }
    };
    auto store = [&](int b) {
        if (t < LW * kQ) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                *(f4a*)&lds[(4 * b + 2 * j) * SZ + 4 * t] = pr[j] * vv;
                *(f4a*)&lds[(4 * b + 2 * j + 1) * SZ + 4 * t] = pw[j];
            }
        }
    };
    fetch(0);

    // The thread's offsets e0 .. e0 + NG - 1, four rows and two columns.
    const int e0 = __builtin_amdgcn_readfirstlane(t / 256) * NG, zq = t % kQ, c0 = t % 256 / kQ * kImgCX;
    const bool ok = c0 < kImgTX && z0 + 4 * zq < nzi;
    const unsigned o0 = 4u * (unsigned)((x0 + c0) * a.nz + FAT + z0 + 4 * zq), cs = 4u * (unsigned)a.nz;
    f4 m[NG][kImgCX];
#pragma unroll
    for (int q = 0; q < NG; ++q)
#pragma unroll
        for (int c = 0; c < kImgCX; ++c) {
            m[q][c] = (f4)0.f;
            if (e0 + q < ne && ok && x0 + c0 + c < xEnd) m[q][c] = ld4(img + nzx * (e0 + q), o0 + c * cs);
        }
    store(0);
    __syncthreads();
    // Offset e0 + q at column c: R window entry c + q, from staged column c0 +
    // e0 on, and W window entry c - q + NG - 1 (for offsets beyond the last,
    // which are not stored, that may lie before the first staged column, in R).
    const int jr = (c0 + e0) * kTZ + 4 * zq, jw = SZ + (c0 + 2 * hExt - e0 - NG + 1) * kTZ + 4 * zq;
    for (int s = 0; s < a.nk; s += 2) {
        if (s + 2 < a.nk) fetch(s + 2);
        if (ok) {
            for (int j = 0; j < 2 && s + j < a.nk; ++j) {
                const float* r = &lds[((s & 2) * 2 + 2 * j) * SZ + jr];
                const float* w = &lds[((s & 2) * 2 + 2 * j) * SZ + jw];
                f4a rw[NG + kImgCX - 1], ww[NG + kImgCX - 1];
#pragma unroll
                for (int i = 0; i < NG + kImgCX - 1; ++i) {
                    rw[i] = *(const f4a*)(r + i * kTZ);
                    ww[i] = *(const f4a*)(w + i * kTZ);
                }
#pragma unroll
                for (int q = 0; q < NG; ++q)
#pragma unroll
                    for (int c = 0; c < kImgCX; ++c) m[q][c] += rw[c + q] * ww[c - q + NG - 1];
            }
        }
        if (s + 2 < a.nk) store((s & 2) ? 0 : 1);
        __syncthreads();
    }
    // The store addresses are formed again here rather than kept live across
    // the sample loop from the loads above.
    unsigned oEnd = o0;
    int eEnd = e0;
    asm volatile("" : "+v"(oEnd), "+v"(eEnd));
    gf* out = img + nzx * __builtin_amdgcn_readfirstlane(eEnd);
#pragma unroll
    for (int q = 0; q < NG; ++q)
#pragma unroll
        for (int c = 0; c < kImgCX; ++c)
            if (e0 + q < ne && ok && x0 + c0 + c < xEnd) st4(out + nzx * q, oEnd + c * cs, m[q][c]);
}

template <bool TOMO>
hipError_t launch(const ExtBatchArgs& a, int nshots, hipStream_t s)
{
    const int nzi = a.nz - 2 * FAT, nxi = a.nx - 2 * FAT;
    if (a.nk < 1 || a.nk > kExtBatchMax || a.hExt < 0 || a.hExt > kOffsetSsMax || !wide_grid_ok(a.nz, a.nx))
        return hipErrorInvalidValue;
    if (nzi <= 0 || nxi <= 0 || nshots < 1) return hipSuccess;
    const int bx = (nxi + kTX - 1) / kTX, bz = (nzi + kTZ - 1) / kTZ, by = (nshots + kShots - 1) / kShots;
    const dim3 g((bx * bz * by + 7) / 8 * 8), n(kThreads);
    hipLaunchKernelGGL((k_offset_ss<kOffsetSsMax, TOMO>), g, n, 0, s, a, nshots, bx, bz, by);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_offset_ss(const ExtBatchArgs& a, int nshots, hipStream_t s) { return launch<false>(a, nshots, s); }
hipError_t launch_offset_ss_tomo(const ExtBatchArgs& a, int nshots, hipStream_t s) { return launch<true>(a, nshots, s); }

hipError_t launch_offset_img(const TimeBatchArgs& a, int nshots, hipStream_t s)
{
    const int nzi = a.nz - 2 * FAT, nxr = a.nx - 2 * FAT - 2 * a.hExt;
    if (a.nk < 1 || a.nk > kTimeBatchMax || a.hExt < 0 || a.hExt > kOffsetSsMax || !wide_grid_ok(a.nz, a.nx))
        return hipErrorInvalidValue;
    if (nzi <= 0 || nxr <= 0 || nshots < 1) return hipSuccess;
    const int bx = (nxr + kImgTX - 1) / kImgTX, bz = (nzi + kTZ - 1) / kTZ;
    const dim3 g((bx * bz * nshots + 7) / 8 * 8);
    hipLaunchKernelGGL((k_offset_img<kOffsetSsMax, 7>), g, dim3(kImgThreads), 0, s, a, bx, bz, nshots);
    return hipGetLastError();
}

}  // namespace aiso
