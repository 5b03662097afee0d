// wide.hip -- the fused time step with four z-points per lane.
//
// One fine time step of a batch of shots, like k_step_generic of kernels.hip
// and in the same arithmetic (the reference's launches it replaces and the
// fused sponge are described there), with the work laid out for wide memory
// operations: a workgroup owns a TZ x TX tile of interior points, each thread
// four consecutive z-points in each of PX consecutive columns, so slices move
// in 16-byte loads and stores and the stencil reads LDS in 16-byte rows.
//
// What bounds it: the memory path.  A step reads two slices and v2dt2 and
// writes one, 16 bytes per point; with the stencil cut to two terms the step
// of 20 shots of 608 x 1312 points still takes 36.4 of its 38.8 us (411
// Gpts/s; one point per lane 44.6 us, 357).  A streaming loop with the same
// accesses moves 500 Gpts/s with 16-byte lanes and 450 with 4-byte ones.
//
// Tiles: 64 rows make four full 256-byte runs per column and keep the halo
// columns at 1.6 (PX 1, 64 x 16) or 1.3 (PX 2, 64 x 32) of the tile.  PX 2
// reads each LDS row for two columns, which pays where two fields share the
// launch (Born lockstep, 24 shots of 608 x 1312: 221 ms, PX 1 234, one point
// per lane 238); PX 1 makes twice the workgroups, which pays for the passes
// of one field (8 shots of 368 x 880 under a free surface, migration: 23.2 ms,
// PX 2 24.4, one point per lane 28.2).
//
// Interior sizes are multiples of 16 (the block size of the padding rule), so
// a thread's points are all inside the grid or all outside it, and no point
// is tested by itself.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "wide.hpp"

namespace aiso {

namespace {

// The tile and its staged copy: LDS column c holds grid column x0 - FAT + c of
// the interior, rows -5 .. TZ + 4 at [kOff + row]; kOff keeps the tile's rows
// 16-byte aligned.
template <int TZ, int PX>
struct WideShape {
    static constexpr int ZL = TZ / 4, XG = NT / ZL, TX = XG * PX;
    static constexpr int kOff = 8, LZ = TZ + 16, LX = TX + 2 * FAT;
    static constexpr int Q = ZL + 2;                        // quads staged per column: rows -4 .. TZ + 3
    static constexpr int KQ = (LX * Q + NT - 1) / NT;       // staged quads per thread
    static_assert(2 * LX <= NT, "one thread per single row element");
};

// What a field's step reads and writes: its slices, and the element offsets
// in W of the samples it uses.
struct Field {
    cgf* pc;
    gf* po;
    long wA, wB;
};

template <int TZ, int PX, unsigned MODE, bool SPONGE, bool FS>
__device__ __forceinline__ void wide_block(const StepArgs& a, const ShotSlot& S, const Field& F, int tile, float* sC)
{
    using T = WideShape<TZ, PX>;
    constexpr int LZ = T::LZ;
    constexpr bool ADJ = MODE & M_ADJ;
    constexpr bool PRE_SPARSE = MODE & (M_INJ_SIG | M_INJ_DATA);
    constexpr bool POST_SPARSE = MODE & (M_REC_DATA | M_REC_SIG);
    constexpr bool WIN = MODE & M_WIN;
    constexpr bool SSB = MODE & M_SS_BORN, SSP = MODE & M_SS_PRE, HAS_SS = SSB || SSP;

    const int nz = a.nz, nx = a.nx, t = threadIdx.x;
    const int z0 = (tile % a.tilesZ) * TZ, x0 = (tile / a.tilesZ) * T::TX;      // interior coordinates
    const int nrow = imin(TZ, nz - 2 * FAT - z0), ncol = imin(T::TX, nx - 2 * FAT - x0);
    const int zq = t % T::ZL, g = t / T::ZL;
    const bool ok = 4 * zq < nrow && PX * g < ncol;
    const unsigned cs = 4u * (unsigned)nz;                                      // column stride in bytes
    const int gz = FAT + z0 + 4 * zq, gx = FAT + x0 + PX * g;                   // the thread's first point
    const unsigned off0 = 4u * (unsigned)(gx * nz + gz);
    cgf* V = G(a.v2dt2);
    const bool useB = a.fb != 0.f;

    // Staging loads first: every wait for them leaves the operand loads
    // issued after them in flight.
    f4 tv[T::KQ], tm[ADJ ? T::KQ : 1];
    int li[T::KQ];
#pragma unroll
    for (int k = 0; k < T::KQ; ++k) {
        const int i = t + k * NT, col = i / T::Q, q = i - col * T::Q - 1;
        const bool in = col < ncol + 2 * FAT && 4 * q <= nrow;
        li[k] = in ? col * LZ + T::kOff + 4 * q : -1;
        const unsigned o = 4u * (unsigned)((x0 + col) * nz + FAT + z0 + 4 * q);
        if (in) {
            tv[k] = ld4(F.pc, o);
            if constexpr (ADJ) tm[k] = ld4(V, o);
        }
    }
    float t1 = 0.f, m1 = 0.f;                                                   // the rows -5 and nrow + 4
    int l1 = -1;
    {
        const int col = t >> 1, row = (t & 1) ? nrow + 4 : -FAT;
        if (col < ncol + 2 * FAT) {
            l1 = col * LZ + T::kOff + row;
            const unsigned o = 4u * (unsigned)((x0 + col) * nz + FAT + z0 + row);
            t1 = *at1(F.pc, o);
            if constexpr (ADJ) m1 = *at1(V, o);
        }
    }

    // Per-point operands, and the sponge factors (their table is read at the
    // distance to the nearest edge; FS: no sponge at the surface,
    // dampCosineEdgeFs, F/src/kernelsGpu.cu:221-239).
    f4 os[PX], pv[PX], dmp[SPONGE ? PX : 1];
    f4 sA[HAS_SS ? PX : 1], sB[HAS_SS ? PX : 1], mm[SSB ? PX : 1];
    cgf* ssa = nullptr;
    cgf* ssb = nullptr;
    f4 gw[(MODE & M_GRAD) ? PX : 1], gi[(MODE & M_GRAD) ? PX : 1];
    if constexpr (HAS_SS) {
        ssa = G(S.W) + F.wA;
        if (useB) ssb = G(S.W) + F.wB;
    }
    if (ok) {
#pragma unroll
        for (int j = 0; j < PX; ++j) {
            const unsigned o = off0 + j * cs;
            os[j] = ld4(F.po, o);
            pv[j] = ld4(ADJ ? F.pc : V, o);
            if constexpr (SSB) mm[j] = ld4(G(a.mtil), o);
            if constexpr (HAS_SS) {
                sA[j] = ld4s(ssa, o, SSP && a.ntW);
                if (useB) sB[j] = ld4s(ssb, o, SSP && a.ntW);
            }
            if constexpr (MODE & M_GRAD) {
                gw[j] = ld4s(G(S.W) + a.wImg, o, a.ntW);
                gi[j] = ld4(G(S.img), o);
            }
            if constexpr (SPONGE) {
                const int dx = imin(gx + j - FAT, nx - 1 - FAT - gx - j);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int db = nz - 1 - FAT - gz - r, d = imin(dx, FS ? db : imin(gz + r - FAT, db));
                    dmp[j][r] = d < a.minPad ? G(a.cd)[d] : 1.f;
                }
            }
        }
    }

#pragma unroll
    for (int k = 0; k < T::KQ; ++k)
        if (li[k] >= 0) *(f4a*)&sC[li[k]] = ADJ ? tv[k] * tm[k] : tv[k];
    if (l1 >= 0) sC[l1] = ADJ ? t1 * m1 : t1;
    __syncthreads();
    if constexpr (FS && !ADJ) {
        // Free surface (setFsConditionFwdGpu, F/src/kernelsGpu.cu:555-567) on
        // a top tile's staged copy, for the interior columns: the surface row
        // is zero and the rows above mirror the rows below with the opposite
        // sign.
        if (z0 == 0) {
            const int c = x0 + t;                                               // grid column of LDS column t
            if (t < ncol + 2 * FAT && c >= FAT && c < nx - FAT) {
                float* col = &sC[t * LZ + T::kOff];
                col[0] = 0.f;
#pragma unroll
                for (int k = 1; k <= FAT; ++k) col[-k] = -col[k];
            }
            __syncthreads();
        }
    }

    const bool surf = FS && z0 == 0 && zq == 0;                                 // the thread's first row is the surface
    f4 nv[PX], cur[WIN ? PX : 1], lv[(MODE & M_LAP) ? PX : 1];
    if (ok) {
        f4a w[PX + 2 * FAT];
#pragma unroll
        for (int i = 0; i < PX + 2 * FAT; ++i) w[i] = *(const f4a*)&sC[(PX * g + i) * LZ + T::kOff + 4 * zq];
#pragma unroll
        for (int j = 0; j < PX; ++j) {
            // e[i]: row i - 5 of the column relative to the thread's first
            const float* s = &sC[(PX * g + j + FAT) * LZ + T::kOff + 4 * zq];
            const f4a up = *(const f4a*)(s - 4), dn = *(const f4a*)(s + 4);
            const float e[14] = {s[-5], up[0], up[1], up[2], up[3], w[j + FAT][0], w[j + FAT][1], w[j + FAT][2],
                                 w[j + FAT][3], dn[0], dn[1], dn[2], dn[3], s[8]};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // 10th-order Laplacian in the reference's summation order: z terms, then x terms
                const float cc = e[r + 5];
                float lap = a.zc[0] * cc
                          + a.zc[1] * (e[r + 4] + e[r + 6])
                          + a.zc[2] * (e[r + 3] + e[r + 7])
                          + a.zc[3] * (e[r + 2] + e[r + 8])
                          + a.zc[4] * (e[r + 1] + e[r + 9])
                          + a.zc[5] * (e[r + 0] + e[r + 10]);
                if constexpr (FS && ADJ) {
                    // stepAdjFsGpu (F/src/kernelsGpu.cu:613-700): below a free
                    // surface four rows drop the z terms the forward folds onto them
                    const int row = 4 * zq + r;
                    if (z0 == 0 && row >= 1 && row <= 4) {
                        if (row == 1) lap = lap - a.zc[2] * e[r + 5] - a.zc[3] * e[r + 6] - a.zc[4] * e[r + 7] - a.zc[5] * e[r + 8];
                        else if (row == 2) lap = lap - a.zc[3] * e[r + 4] - a.zc[4] * e[r + 5] - a.zc[5] * e[r + 6];
                        else if (row == 3) lap = lap - a.zc[4] * e[r + 3] - a.zc[5] * e[r + 4];
                        else lap = lap - a.zc[5] * e[r + 2];
                    }
                }
                lap = lap
                    + a.xc[0] * cc
                    + a.xc[1] * (w[j + 6][r] + w[j + 4][r])
                    + a.xc[2] * (w[j + 7][r] + w[j + 3][r])
                    + a.xc[3] * (w[j + 8][r] + w[j + 2][r])
                    + a.xc[4] * (w[j + 9][r] + w[j + 1][r])
                    + a.xc[5] * (w[j + 10][r] + w[j + 0][r]);
                if constexpr (MODE & M_LAP) lv[j][r] = lap;
                const bool onSurf = FS && r == 0 && surf;
                // forward: the old slice's surface value reads as zero, as the
                // reference zeroed it when it was the current one
                const float osj = (!ADJ && onSurf) ? 0.f : os[j][r];
                const float o = SPONGE ? osj * dmp[j][r] : osj;                // second damping of the old slice
                float n;
                if constexpr (ADJ) {
                    const float c = pv[j][r];
                    n = onSurf ? o : lap + c + c - o;                           // the adjoint leaves the surface row
                    if constexpr (WIN) cur[j][r] = c;
                } else {
                    n = pv[j][r] * lap + cc + cc - o;
                    // the window takes the slices as stored; at the surface
                    // the staged value is the mirrored one
                    if constexpr (WIN) cur[j][r] = onSurf ? *at1(F.pc, off0 + j * cs) : cc;
                }
                if constexpr (SSB) {
                    const float x = mm[j][r] * sA[j][r];
                    if (useB) n += x * a.fa + (mm[j][r] * sB[j][r]) * a.fb;
                    else n += x * a.fa;
                }
                if constexpr (SSP) {
                    if (useB) n += sA[j][r] * a.fa + sB[j][r] * a.fb;
                    else n += sA[j][r] * a.fa;
                }
                nv[j][r] = n;
            }
        }
    }

    // The tile's sparse entries go through the LDS tile sN [TX][TZ], which
    // takes the staged tile's place once every thread has read it.
    float* sN = sC;
    const int* tp = nullptr;
    if constexpr (PRE_SPARSE) {
        tp = (MODE & M_INJ_SIG) ? S.srcTile : S.recTile;
        const int2* te = (MODE & M_INJ_SIG) ? S.srcEnt : S.recEnt;
        const int e0 = tp[tile], e1 = tp[tile + 1];
        if (e1 > e0) {                                                          // block-uniform
            __syncthreads();
            if (ok) {
#pragma unroll
                for (int j = 0; j < PX; ++j) *(f4a*)&sN[(PX * g + j) * TZ + 4 * zq] = nv[j];
            }
            __syncthreads();
            for (int e = e0 + t; e < e1; e += NT) {
                const int2 en = te[e];
                float v;
                if constexpr (MODE & M_INJ_SIG) {
                    v = G(S.sig)[(long)en.y * a.ntw + a.itwInj];
                } else {
                    cgf* dr = G(S.dreg) + ((long)en.y * a.nts + a.its);
                    v = dr[0] * a.fc + dr[1] * a.fd;
                }
                sN[en.x] += v;
            }
            __syncthreads();
            if (ok) {
#pragma unroll
                for (int j = 0; j < PX; ++j) nv[j] = *(const f4a*)&sN[(PX * g + j) * TZ + 4 * zq];
            }
        }
    }
    int postE0 = 0, postE1 = 0;
    const int2* postTe = nullptr;
    gf* postOut = nullptr;
    if constexpr (POST_SPARSE) {
        const int* rp = (MODE & M_REC_SIG) ? S.srcTile : S.recTile;
        postTe = (MODE & M_REC_SIG) ? S.srcEnt : S.recEnt;
        postOut = G((MODE & M_REC_SIG) ? S.sig : S.dreg);
        postE0 = rp[tile];
        postE1 = rp[tile + 1];
    }

    // The shot's buffers written below, read from its slot before the first
    // store: the compiler cannot tell that the stores leave the slot alone.
    gf* A = nullptr;
    gf* B = nullptr;
    if constexpr (MODE & M_CAPTURE) {
        // forward passes capture the coarse source wavefield W; the adjoint
        // receiver pass accumulates into the two ss slices
        A = G(ADJ ? S.ss[a.ssA] : S.W) + (ADJ ? a.ssOffA : F.wA);
        B = G(ADJ ? S.ss[a.ssB] : S.W) + (ADJ ? a.ssOffB : F.wB);
    }
    gf* lapW = (MODE & M_LAP) ? G(S.W) + F.wA : nullptr;
    gf* gImg = (MODE & M_GRAD) ? G(S.img) : nullptr;
    gf* imgI = nullptr;
    cgf* imgW = nullptr;
    if constexpr (MODE & M_IMAGE) {
        if (a.image) {
            imgI = G(S.img);
            imgW = G(S.W) + a.wImg;
        }
    }
    gf* winDst = nullptr;                                                       // window capture
    cgf* winMul = nullptr;                                                      // WIN_SS: m~; WIN_IMG: the W sample
    if constexpr (WIN) {
        if (a.win) {
            if (a.winOut == WIN_W || a.winOut == WIN_SS) {
                winDst = G(S.W) + F.wA;
                if (a.winOut == WIN_SS) winMul = G(a.mtil);
            } else if (a.winOut == WIN_IMG) {
                winDst = G(S.img);
                winMul = G(S.W) + a.wImg;
            } else {
                winDst = G(S.ss[a.ssA]) + a.ssOffA;
            }
        }
    }
    if (ok) {
#pragma unroll
        for (int j = 0; j < PX; ++j) {
            const unsigned o = off0 + j * cs;
            const f4 n = SPONGE ? nv[j] * dmp[j] : nv[j];
            nv[j] = n;
            if constexpr (MODE & M_CAPTURE) {
                // a zero weight leaves the slice as it is (x + n*0 == x); a
                // first touch writes instead of accumulating into a zeroed slice
                if (!a.skipA) st4(A, o, a.assignA ? n * a.fe : ld4(A, o) + n * a.fe);
                else if (a.assignA) st4(A, o, (f4)0.f);
                f4 bnew = (f4)0.f;
                if (!a.skipB) {
                    bnew = a.assignB ? n * a.ff : ld4(B, o) + n * a.ff;
                    st4(B, o, bnew);
                } else if (a.assignB) {
                    st4(B, o, (f4)0.f);
                } else if constexpr (MODE & M_IMAGE) {
                    bnew = ld4(B, o);
                }
                if constexpr (MODE & M_IMAGE) {
                    if (a.image) st4(imgI, o, ld4(imgI, o) + ld4(imgW, o) * bnew);
                }
            }
            if constexpr (WIN) {
                if (a.win) {
                    // coarse sample from three consecutive fine slices, in the
                    // reference's order (old, current, new)
                    const f4 v = (os[j] * a.wa + cur[j] * a.wb) + n * a.wc;
                    switch (a.winOut) {
                    case WIN_W: st4s(winDst, o, v, a.ntW); break;
                    case WIN_SS: st4s(winDst, o, ld4(winMul, o) * v, a.ntW); break;
                    case WIN_IMG: st4(winDst, o, ld4(winDst, o) + ld4s(winMul, o, a.ntW) * v); break;
                    default: st4(winDst, o, v); break;
                    }
                }
            }
            if constexpr (MODE & M_LAP) st4s(lapW, o, lv[j], a.ntW);
            if constexpr (MODE & M_GRAD) st4(gImg, o, gi[j] + gw[j] * n);
            st4(F.po, o, n);
        }
    }

    if constexpr (POST_SPARSE) {
        if (postE1 > postE0) {                                                  // block-uniform
            __syncthreads();
            if (ok) {
#pragma unroll
                for (int j = 0; j < PX; ++j) *(f4a*)&sN[(PX * g + j) * TZ + 4 * zq] = nv[j];
            }
            __syncthreads();
            for (int e = postE0 + t; e < postE1; e += NT) {
                const int2 en = postTe[e];
                const float n = sN[en.x];
                if constexpr (MODE & M_REC_SIG) {
                    postOut[(long)en.y * a.ntw + a.itwRec] += n;
                } else {
                    gf* dr = postOut + ((long)en.y * a.nts + a.its);
                    dr[0] += n * a.fe;
                    dr[1] += n * a.ff;
                }
            }
        }
    }
}

// Whether the sponge reaches a tile (block-uniform).
template <int TZ, int TX, bool FS>
__device__ __forceinline__ bool tile_in_sponge(const StepArgs& a, int tile)
{
    const int z0 = (tile % a.tilesZ) * TZ, x0 = (tile / a.tilesZ) * TX;
    const int nzi = a.nz - 2 * FAT, nxi = a.nx - 2 * FAT;
    const int dz = imin(FS ? a.minPad : z0, nzi - imin(nzi, z0 + TZ)), dx = imin(x0, nxi - imin(nxi, x0 + TX));
    return imin(dz, dx) < a.minPad;
}

template <int TZ, int PX, unsigned MODE, bool FS>
__device__ __forceinline__ void wide_tile(const StepArgs& a, const ShotSlot& S, const Field& F, int tile, float* sC)
{
    if (tile_in_sponge<TZ, WideShape<TZ, PX>::TX, FS>(a, tile)) wide_block<TZ, PX, MODE, true, FS>(a, S, F, tile, sC);
    else wide_block<TZ, PX, MODE, false, FS>(a, S, F, tile, sC);
}

template <int TZ, int PX, unsigned MODE, bool FS>
__global__ __launch_bounds__(NT) void k_wide(const StepArgs a)
{
    using T = WideShape<TZ, PX>;
    __shared__ __attribute__((aligned(16))) float sC[T::LX * T::LZ];
    const int logical = xcd_logical(blockIdx.x, gridDim.x);
    if (logical >= a.gridLogical) return;                                       // padding blocks (block-uniform)
    const int shot = logical / a.ntiles, tile = logical - shot * a.ntiles;
    const ShotSlot& S = a.slots[shot];
    wide_tile<TZ, PX, MODE, FS>(a, S, Field{G(S.p[a.cur]), G(S.p[a.cur ^ 1]), a.wA, a.wB}, tile, sC);
}

// Lockstep Born forward, sub == 2 (k_fwd_pair of kernels.hip): the source
// field's step t and the scattered field's step t - 2 in one launch, as two
// workgroups per tile that run side by side and share v2dt2 in L2.
template <int TZ, int PX, bool FS>
__global__ __launch_bounds__(NT) void k_wide_pair(const StepArgs a)
{
    using T = WideShape<TZ, PX>;
    __shared__ __attribute__((aligned(16))) float sC[T::LX * T::LZ];
    const int logical = xcd_logical(blockIdx.x, gridDim.x);
    if (logical >= 2 * a.gridLogical) return;                                   // padding blocks (block-uniform)
    const int unit = logical >> 1, shot = unit / a.ntiles, tile = unit - shot * a.ntiles;
    const ShotSlot& S = a.slots[shot];
    if (logical & 1)
        wide_tile<TZ, PX, MODE_BORN_SCAT_PRE, FS>(a, S, Field{G(S.q[a.curQ]), G(S.q[a.curQ ^ 1]), a.wQa, a.wQb}, tile, sC);
    else
        wide_tile<TZ, PX, MODE_SRC_WIN, FS>(a, S, Field{G(S.p[a.cur]), G(S.p[a.cur ^ 1]), a.wA, a.wB}, tile, sC);
}

using WideKernel = void (*)(const StepArgs);

hipError_t launch(WideKernel k, int blocks, const StepArgs& a, hipStream_t s, hipEvent_t e0, hipEvent_t e1)
{
    const dim3 grid((blocks + 7) / 8 * 8);
    if (e0 && e1) hipExtLaunchKernelGGL(k, grid, dim3(NT), 0, s, e0, e1, 0, a);
    else hipLaunchKernelGGL(k, grid, dim3(NT), 0, s, a);
    return hipGetLastError();
}

}  // namespace

static_assert(WideShape<kWideTZ, 1>::TX == kWideTX && WideShape<kWideTZ, 2>::TX == kWidePairTX, "tile widths");

// 16-point blocks (a thread's points are inside or outside together) and
// 32-bit byte offsets within a slice.
bool wide_grid_ok(int nz, int nx)
{
    return (nz - 2 * FAT) % 16 == 0 && (nx - 2 * FAT) % 16 == 0 && (long)nz * nx < (1L << 30);
}

hipError_t launch_wide(unsigned mode, int tx, const StepArgs& a, hipStream_t s, hipEvent_t e0, hipEvent_t e1)
{
    if (!wide_grid_ok(a.nz, a.nx)) return hipErrorInvalidValue;
    WideKernel k = nullptr;
    if (tx == kWidePairTX) {
        switch (mode) {
        case MODE_SRC_WIN: k = a.fs ? (WideKernel)k_wide<kWideTZ, 2, MODE_SRC_WIN, true> : k_wide<kWideTZ, 2, MODE_SRC_WIN, false>; break;
        case MODE_BORN_SCAT_PRE:
            k = a.fs ? (WideKernel)k_wide<kWideTZ, 2, MODE_BORN_SCAT_PRE, true> : k_wide<kWideTZ, 2, MODE_BORN_SCAT_PRE, false>;
            break;
        }
    } else if (tx == kWideTX && a.fs) {
        switch (mode) {
        case MODE_NL_FWD: k = k_wide<kWideTZ, 1, MODE_NL_FWD, true>; break;
        case MODE_NL_ADJ: k = k_wide<kWideTZ, 1, MODE_NL_ADJ, true>; break;
        case MODE_SRC: k = k_wide<kWideTZ, 1, MODE_SRC, true>; break;
        case MODE_SRC_WIN: k = k_wide<kWideTZ, 1, MODE_SRC_WIN, true>; break;
        case MODE_BORN_SCAT: k = k_wide<kWideTZ, 1, MODE_BORN_SCAT, true>; break;
        case MODE_BORN_SCAT_PRE: k = k_wide<kWideTZ, 1, MODE_BORN_SCAT_PRE, true>; break;
        case MODE_BORN_REC: k = k_wide<kWideTZ, 1, MODE_BORN_REC, true>; break;
        case MODE_REC_WIN: k = k_wide<kWideTZ, 1, MODE_REC_WIN, true>; break;
        }
    } else if (tx == kWideTX) {
        switch (mode) {
        case MODE_NL_FWD: k = k_wide<kWideTZ, 1, MODE_NL_FWD, false>; break;
        case MODE_NL_ADJ: k = k_wide<kWideTZ, 1, MODE_NL_ADJ, false>; break;
        case MODE_SRC: k = k_wide<kWideTZ, 1, MODE_SRC, false>; break;
        case MODE_SRC_LAP: k = k_wide<kWideTZ, 1, MODE_SRC_LAP, false>; break;
        case MODE_ADJ_GRAD: k = k_wide<kWideTZ, 1, MODE_ADJ_GRAD, false>; break;
        }
    }
    if (!k) return hipErrorInvalidValue;
    StepArgs b = a;
    b.gridLogical = a.ntiles * a.nshots;                                        // one workgroup per (tile, shot)
    return launch(k, b.gridLogical, b, s, e0, e1);
}

hipError_t launch_wide_pair(const StepArgs& a, hipStream_t s, hipEvent_t e0, hipEvent_t e1)
{
    if (!wide_grid_ok(a.nz, a.nx)) return hipErrorInvalidValue;
    WideKernel k = a.fs ? (WideKernel)k_wide_pair<kWideTZ, 2, true> : k_wide_pair<kWideTZ, 2, false>;
    StepArgs b = a;
    b.gridLogical = a.ntiles * a.nshots;
    return launch(k, 2 * b.gridLogical, b, s, e0, e1);
}

}  // namespace aiso
