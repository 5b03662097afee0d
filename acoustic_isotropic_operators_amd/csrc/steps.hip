// steps.hip -- several fine time steps of a pass per launch: the nonlinear and
// Born passes and those of the velocity gradient.
//
// Passes over few points are bound by launches: a one-step launch takes the
// host 3.9 us to submit and the GPU 4.1 us for 304 x 512 points, most of it
// launch and memory latency.  Here a workgroup copies a tile and a halo of K
// stencils into LDS, advances it K steps, each on the region the next one
// still needs, and writes the tile's two newest slices to the field's other
// pair of slices (its neighbours read the old pair).  Sources inject and
// receivers record inside the launch; the points are updated in the order of
// operations of the one-step kernels.
//
// What bounds it: the latency of K dependent steps, each a pass over LDS with
// 16 waves per CU and a barrier; the halo's redundant points (62 x 62 for a
// 32 x 32 tile's first of 4 steps) run in lanes that would idle.  Per step of
// the nonlinear forward / adjoint on MI355X, no sources or receivers (one-step
// launches on one lane or two: 4.1 us for 1 shot, 6.9-7.4 us from 2 shots on):
//   304 x 512 points, 1 shot:   32 x 32 tiles, 4 steps   2.11 / 2.25 us
//                    3 shots:   64 x 32 tiles, 3 steps   2.71 / 2.86 us
//                    6 shots:   64 x 64 tiles, 3 steps   3.45 / 3.80 us
// A source and 400 receivers add 0.5 us per step to the first: the tiles that
// hold them take longer, and all tiles run at once.  The smallest tile whose
// workgroups all run at once (one per CU) is best: 3 shots on 32 x 32 tiles
// take 3.75 us, 1 shot on 64 x 64 tiles 3.22.  Over many workgroups the
// one-step kernels, which are bound by memory and not by latency, are faster
// (16 shots of 608 x 1312 points: 411 Gpts/s against 371), but for the passes
// that also move an image or a slice of W at every step: here they move once
// per launch, held by one thread per quad of the tile (gradient of 8 shots of
// 512 x 1104 points: 37 us per step of both fields, one-step launches 49).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "wide.hpp"

namespace aiso {

namespace {

constexpr int kFew = 4;    // injecting points that the computing threads look for

template <int N>
struct IC {
    static constexpr int v = N;
};

// Value that sparse entry (.., trace y) adds at step i: a column of sig, or
// the data samples its, its + 1 with their weights.
template <bool ADJ>
__device__ __forceinline__ float injected(const StepsArgs& a, const ShotSlot& S, int y, int i)
{
    if constexpr (ADJ) {
        cgf* d = G(S.dreg) + ((long)y * a.nts + a.its[i]);
        return d[0] * a.wi[i][0] + d[1] * a.wi[i][1];
    } else {
        return G(S.sig)[(long)y * a.ntw + a.itw[i]];
    }
}

template <int TZ, int TX, int K, int NTH, int PX, unsigned MODE>
__global__ __launch_bounds__(NTH) void k_steps(const StepsArgs a)
{
    using T = StepsShape<TZ, TX, K>;
    constexpr bool ADJ = MODE & M_ADJ, REC = MODE & (M_REC_DATA | M_REC_SIG);
    // OWN: each thread keeps a quad of the tile's points over the steps
    constexpr bool WIN = MODE & M_WIN, CAP = MODE & M_CAPTURE, OWN = (MODE & M_GRAD) || WIN || CAP;
    constexpr bool SSB = MODE & M_SS_BORN, SSP = MODE & M_SS_PRE;
    constexpr bool INJ = MODE & (M_INJ_SIG | M_INJ_DATA);
    static_assert(TZ / 4 * TX <= NTH, "a thread per quad of the tile");
    constexpr int E = T::E, HZ = T::HZ, LZ = T::LZ, SZ = T::SZ;
    __shared__ __attribute__((aligned(16))) float lds[steps_slices(ADJ) * SZ + kStepsPadMax + 1];
    __shared__ int fewI[kFew];
    __shared__ float fewV[K][kFew];
    const int t = threadIdx.x, nzi = a.nz - 2 * FAT, nxi = a.nx - 2 * FAT;
    const int l = xcd_logical(blockIdx.x, gridDim.x);
    if (l >= a.ntiles * a.nshots) return;                                       // padding blocks (block-uniform)
    const int shot = l / a.ntiles, tile = l - shot * a.ntiles;
    const ShotSlot& S = a.slots[shot];
    const int z0 = (tile % a.tilesZ) * TZ, x0 = (tile / a.tilesZ) * TX;         // interior coordinates
    auto at = [&](int row, int x) -> unsigned { return 4u * (unsigned)((x + FAT) * a.nz + FAT + row); };

    // The tile and its halo of E points, zero outside the interior: the two
    // slices (step ks of K reads slice ks & 1 and overwrites the other), and
    // v2dt2 or the adjoint's products v2dt2 * slice, which its stencil reads.
    float* const P0 = lds;
    float* const P1 = lds + SZ;
    float* const V0 = lds + 2 * SZ;
    float* const V1 = lds + 3 * SZ;
    float* const cd = lds + steps_slices(ADJ) * SZ;                             // sponge factors, 1 past the last
    const bool odd = (K - a.n) & 1;                                             // parity of the launch's first step
    gf* Cn = G(S.p[2 * (a.pair ^ 1)]);                                          // the two newest slices go to the other pair
    gf* On = G(S.p[2 * (a.pair ^ 1) + 1]);
    cgf* VG = G(a.v2dt2);
    // Sparse entries: those of the region inject, those of the tile record.
    const int i0 = INJ ? (ADJ ? S.recTile : S.srcTile)[tile] : 0;
    const int i1 = INJ ? (ADJ ? S.recTile : S.srcTile)[tile + 1] : 0;
    const int r0 = REC ? (ADJ ? S.srcOwnTile : S.recOwnTile)[tile] : 0;
    const int r1 = REC ? (ADJ ? S.srcOwnTile : S.recOwnTile)[tile + 1] : 0;
    {
        cgf* C = G(S.p[2 * a.pair]);
        cgf* O = G(S.p[2 * a.pair + 1]);
        constexpr int QC = (TZ + 2 * HZ) / 4, U = QC * T::XC, KU = (U + NTH - 1) / NTH;
        f4 c[KU], o[KU], v[KU];
        int li[KU];
#pragma unroll
        for (int k = 0; k < KU; ++k) {
            const int u = t + k * NTH, col = u / QC, q = u - col * QC, x = x0 - E + col, row = z0 - HZ + 4 * q;
            li[k] = u < U ? T::index(row - z0, x - x0) : -1;
            c[k] = o[k] = v[k] = (f4)0.f;
            if (u < U && x >= 0 && x < nxi && row >= 0 && row < nzi) {
                const unsigned off = at(row, x);
                c[k] = ld4(C, off);
                v[k] = ld4(VG, off);
                o[k] = ld4(O, off);
            }
        }
        for (int i = t; i <= a.minPad; i += NTH) cd[i] = i < a.minPad ? G(a.cd)[i] : 1.f;
#pragma unroll
        for (int k = 0; k < KU; ++k)
            if (li[k] >= 0) {
                *(f4a*)&P0[li[k]] = odd ? o[k] : c[k];
                *(f4a*)&P1[li[k]] = odd ? c[k] : o[k];
                if constexpr (ADJ) {
                    *(f4a*)&V0[li[k]] = odd ? (f4)0.f : c[k] * v[k];
                    *(f4a*)&V1[li[k]] = odd ? c[k] * v[k] : (f4)0.f;
                } else {
                    *(f4a*)&V0[li[k]] = v[k];
                }
            }
    }
    // The thread's quad of the tile, and what it holds over the steps: the image
    // and the samples of W it is made from; the quad's old and current values
    // for the window capture; the two samples of W that a capture adds to.
    const int oq = t % (TZ / 4), oc = t / (TZ / 4), oli = T::index(4 * oq, oc);
    const bool own = OWN && t < TZ / 4 * TX && z0 + 4 * oq < nzi && x0 + oc < nxi;
    const unsigned ooff = own ? at(z0 + 4 * oq, x0 + oc) : 0u;
    constexpr bool IMG = (MODE & M_GRAD) || (WIN && ADJ);
    constexpr int NW = (MODE & M_GRAD) ? K : (K + 1) / 2;                       // windows: every other step at most
    f4 img = (f4)0.f, ow[IMG ? NW : 1], mt = (f4)1.f, ro, rc, cA, cB;
    if (own) {
        if constexpr (IMG) {
            img = ld4(G(S.img), ooff);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if (k >= a.n) continue;
                if constexpr (MODE & M_GRAD) ow[k] = ld4s(G(S.W) + (a.wOff - k * a.wStep), ooff, a.ntW);
                else if (a.first[k]) ow[k / 2] = ld4s(G(S.W) + (a.its[k] + 1) * a.wStep, ooff, a.ntW);
            }
        }
        if constexpr (WIN) {
            // from memory: the LDS copy of the old slice is overwritten by the
            // first step, in other threads, with no barrier before it
            ro = ld4(G(S.p[2 * a.pair + 1]), ooff);
            rc = ld4(G(S.p[2 * a.pair]), ooff);
            if constexpr (!ADJ)
                if (a.mtil) mt = ld4(G(a.mtil), ooff);
        }
        if constexpr (CAP) {
            if (!a.first[0] || a.its[0] > 0) cA = ld4(G(S.W) + a.its[0] * a.wStep, ooff);
            if (!a.first[0]) cB = ld4(G(S.W) + (a.its[0] + 1) * a.wStep, ooff);
        }
    }
    // The first NTH entries of each list are held by a thread for all steps.
    const int2* ie = ADJ ? S.recEnt : S.srcEnt;
    const int2* re = ADJ ? S.srcOwnEnt : S.recOwnEnt;
    // Few injecting points (a source) are added by the threads that compute
    // them; more (a line of receivers) between the step and its sponge.
    const int few = i1 - i0 <= kFew ? i1 - i0 : 0;
    const bool inj = i1 > i0 && !few, rec = r1 > r0;
    int ii = -1, ri = -1;
    float iv[K], rv[K];
#pragma unroll
    for (int k = 0; k < K; ++k) iv[k] = rv[k] = 0.f;
    if (i0 + t < i1) {
        const int2 en = ie[i0 + t];
        ii = en.x;
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (k < a.n) iv[k] = injected<ADJ>(a, S, en.y, k);
        if (t < few) {
            fewI[t] = ii;
#pragma unroll
            for (int k = 0; k < K; ++k) fewV[k][t] = iv[k];
        }
    }
    // a recorder's cells: its ascends by at most one per step, so samples
    // its[0] .. its[0] + K; the adjoint's are columns of sig
    gf* rd = nullptr;
    constexpr int NA = ADJ ? K : K + 1;
    float acc[NA];
    const int last = ADJ ? a.n - 1 : a.its[a.n - 1] - a.its[0] + 1;
    if (r0 + t < r1) {
        const int2 en = re[r0 + t];
        ri = en.x;
        rd = ADJ ? G(S.sig) + ((long)en.y * a.ntw + a.itw[0]) : G(S.dreg) + ((long)en.y * a.nts + a.its[0]);
#pragma unroll
        for (int j = 0; j < NA; ++j)
            if (j <= last) acc[j] = rd[ADJ ? -j : j];
    }
    __syncthreads();
    const bool sponge = z0 - HZ < a.minPad || x0 - E < a.minPad || z0 + TZ + HZ > nzi - a.minPad || x0 + TX + E > nxi - a.minPad;

    auto step = [&](auto KS, auto SPONGE) {
        // step ks of K from the halo's outer edge: its region is the tile and e points around it
        constexpr int ks = decltype(KS)::v;
        constexpr bool LAST = ks == K - 1;
        constexpr int e = FAT * (K - 1 - ks), hz = steps_up4(e);
        constexpr int UQ = (TZ + 2 * hz) / 4, UC = (TX + 2 * e + PX - 1) / PX, U = UQ * UC;
        const int i = ks - (K - a.n);                                           // step of the launch
        if (i < 0) return;                                                      // fewer steps than K (uniform)
        const float* const cur = ks & 1 ? P1 : P0;
        float* const old = ks & 1 ? P0 : P1;                                    // becomes the new slice
        const float* const prod = ks & 1 ? V1 : V0;
        float* const prodN = ks & 1 ? V0 : V1;
        // sponge factors of four rows of a column
        auto damp = [&](int row, int x) {
            const int dx = imin(x, nxi - 1 - x);
            f4 d;
#pragma unroll
            for (int r = 0; r < 4; ++r) d[r] = cd[imin(a.minPad, imin(dx, imin(row + r, nzi - 1 - row - r)))];
            return d;
        };
        auto each = [&](auto f) {
            for (int u = t; u < U; u += NTH) {
                const int g = u / UQ, q = u - g * UQ, c = PX * g - e, row = 4 * q - hz;   // relative to the tile
                if (z0 + row >= 0 && z0 + row < nzi) f(row, c);
            }
        };
        const float* src = ADJ ? prod : cur;
        each([&](int row, int c) {
            const float* s = src + T::index(row, c);
            f4a w[PX + 2 * FAT];
#pragma unroll
            for (int k = 0; k < PX + 2 * FAT; ++k) w[k] = *(const f4a*)(s + (k - FAT) * LZ);
#pragma unroll
            for (int j = 0; j < PX; ++j) {
                if (x0 + c + j < 0 || x0 + c + j >= nxi) continue;
                const float* sj = s + j * LZ;
                const int li = T::index(row, c + j);
                f4 sA, sB;                                                      // secondary source
                if constexpr (SSB || SSP) {
                    const unsigned off = at(z0 + row, x0 + c + j);
                    cgf* W = G(S.W) + a.its[i] * a.wStep;
                    sA = ld4(W, off);
                    if (a.fb[i] != 0.f) sB = ld4(W + a.wStep, off);
                    if constexpr (SSB) {
                        const f4 m = ld4(G(a.mtil), off);
                        sA = m * sA;
                        if (a.fb[i] != 0.f) sB = m * sB;
                    }
                }
                const f4a up = *(const f4a*)(sj - 4), dn = *(const f4a*)(sj + 4), m = w[j + FAT];
                const float z[14] = {sj[-5], up[0], up[1], up[2], up[3], m[0], m[1], m[2], m[3], dn[0], dn[1], dn[2], dn[3], sj[8]};
                f4 o = *(const f4a*)&old[li];
                f4 v;
                if constexpr (ADJ) v = ld4(VG, at(z0 + row, x0 + c + j));
                else v = *(const f4a*)&V0[li];
                f4 cc = m;
                if constexpr (ADJ) cc = *(const f4a*)&cur[li];
                f4 d = (f4)1.f;
                if constexpr (SPONGE.v) d = damp(z0 + row, x0 + c + j);
                f4 n, la;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    // 10th-order Laplacian in the reference's summation order: z terms, then x terms
                    const float lap = a.zc[0] * z[r + 5]
                                    + a.zc[1] * (z[r + 4] + z[r + 6])
                                    + a.zc[2] * (z[r + 3] + z[r + 7])
                                    + a.zc[3] * (z[r + 2] + z[r + 8])
                                    + a.zc[4] * (z[r + 1] + z[r + 9])
                                    + a.zc[5] * (z[r + 0] + z[r + 10])
                                    + a.xc[0] * z[r + 5]
                                    + a.xc[1] * (w[j + 6][r] + w[j + 4][r])
                                    + a.xc[2] * (w[j + 7][r] + w[j + 3][r])
                                    + a.xc[3] * (w[j + 8][r] + w[j + 2][r])
                                    + a.xc[4] * (w[j + 9][r] + w[j + 1][r])
                                    + a.xc[5] * (w[j + 10][r] + w[j + 0][r]);
                    const float od = SPONGE.v ? o[r] * d[r] : o[r];            // second damping of the old slice
                    if constexpr (MODE & M_LAP) la[r] = lap;
                    if constexpr (ADJ) n[r] = lap + cc[r] + cc[r] - od;
                    else n[r] = v[r] * lap + cc[r] + cc[r] - od;
                }
                if constexpr (SSB || SSP) {
                    if (a.fb[i] != 0.f) n += sA * a.fa[i] + sB * a.fb[i];
                    else n += sA * a.fa[i];
                }
                if constexpr (MODE & M_LAP)
                    if (LAST || (row >= 0 && row < TZ && c + j >= 0 && c + j < TX))
                        st4s(G(S.W) + (a.wOff + i * a.wStep), at(z0 + row, x0 + c + j), la, a.ntW);
                for (int k = 0; k < few; ++k) {
                    const int r = fewI[k] - li;
                    if (r >= 0 && r < 4) n[r] += fewV[i][k];
                }
                if constexpr (SPONGE.v)
                    if (!inj) n = n * d;
                if constexpr (LAST) {
                    if (!inj) {
                        const unsigned off = at(z0 + row, x0 + c + j);
                        st4(Cn, off, n);
                        st4(On, off, cc);
                    }
                    if (inj || rec || OWN) *(f4a*)&old[li] = n;
                } else {
                    *(f4a*)&old[li] = n;
                    if constexpr (ADJ)
                        if (!inj) *(f4a*)&prodN[li] = n * v;
                }
            }
        });
        if (inj) {                                                              // block-uniform
            __syncthreads();
            if (ii >= 0) {
                float v = 0.f;
#pragma unroll
                for (int k = 0; k < K; ++k) v = k == i ? iv[k] : v;
                old[ii] += v;
            }
            for (int k = i0 + t + NTH; k < i1; k += NTH) {
                const int2 en = ie[k];
                old[en.x] += injected<ADJ>(a, S, en.y, i);
            }
            __syncthreads();
            if constexpr (SPONGE.v || ADJ || LAST) {
                each([&](int row, int c) {
#pragma unroll
                    for (int j = 0; j < PX; ++j) {
                        if (x0 + c + j < 0 || x0 + c + j >= nxi) continue;
                        const int li = T::index(row, c + j);
                        f4 n = *(const f4a*)&old[li];
                        if constexpr (SPONGE.v) {
                            n = n * damp(z0 + row, x0 + c + j);
                            *(f4a*)&old[li] = n;
                        }
                        if constexpr (LAST) {
                            const unsigned off = at(z0 + row, x0 + c + j);
                            st4(Cn, off, n);
                            st4(On, off, *(const f4a*)&cur[li]);
                        } else if constexpr (ADJ) {
                            *(f4a*)&prodN[li] = n * ld4(VG, at(z0 + row, x0 + c + j));
                        }
                    }
                });
            }
        }
        if (!LAST || rec || OWN) __syncthreads();
        const float* const n = old;
        if constexpr (MODE & M_GRAD) {
            if (own) {
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (k == i) img = img + ow[k] * *(const f4a*)&n[oli];
            }
        }
        if constexpr (WIN) {
            if (own) {
                const f4 nq = *(const f4a*)&n[oli];
                if (a.first[i]) {
                    // coarse sample from three consecutive fine slices, in the
                    // reference's order (old, current, new)
                    f4 v = (ro * a.wa + rc * a.wb) + nq * a.wc;
                    if constexpr (ADJ) {
#pragma unroll
                        for (int k = 0; k < NW; ++k)
                            if (k == i / 2) img = img + ow[k] * v;
                    } else {
                        if (a.mtil) v = mt * v;
                        st4s(G(S.W) + a.its[i] * a.wStep, ooff, v, a.ntW);
                    }
                }
                ro = rc;
                rc = nq;
            }
        }
        if constexpr (CAP) {
            if (own) {
                const f4 nq = *(const f4a*)&n[oli];
                const bool first = a.first[i];                                  // of its coarse interval
                if (first && i > 0) {
                    st4(G(S.W) + (a.its[i] - 1) * a.wStep, ooff, cA);
                    cA = cB;
                }
                // a zero weight leaves the sample as it is; a first touch
                // writes instead of adding to a zeroed one
                const float fe = a.wi[i][0], ff = a.wi[i][1];
                if (fe != 0.f) cA = first && a.its[i] == 0 ? nq * fe : cA + nq * fe;
                else if (first && a.its[i] == 0) cA = (f4)0.f;
                if (ff != 0.f) cB = first ? nq * ff : cB + nq * ff;
                else if (first) cB = (f4)0.f;
            }
        }
        if constexpr (!REC) return;
        if (ri >= 0) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if constexpr (ADJ) acc[k] = k == i ? acc[k] + n[ri] : acc[k];
                else rv[k] = k == i ? n[ri] : rv[k];
            }
        }
        for (int k = r0 + t + NTH; k < r1; k += NTH) {
            const int2 en = re[k];
            if constexpr (ADJ) {
                G(S.sig)[(long)en.y * a.ntw + a.itw[i]] += n[en.x];
            } else {
                gf* d = G(S.dreg) + ((long)en.y * a.nts + a.its[i]);
                d[0] += n[en.x] * a.wi[i][0];
                d[1] += n[en.x] * a.wi[i][1];
            }
        }
    };
    auto all = [&](auto SPONGE) {
        step(IC<0>{}, SPONGE);
        if constexpr (K > 1) step(IC<1>{}, SPONGE);
        if constexpr (K > 2) step(IC<2>{}, SPONGE);
        if constexpr (K > 3) step(IC<3>{}, SPONGE);
    };
    if (sponge) all(IC<1>{});
    else all(IC<0>{});

    if (own) {
        if constexpr (IMG) st4(G(S.img), ooff, img);
        if constexpr (CAP) {
            st4(G(S.W) + a.its[a.n - 1] * a.wStep, ooff, cA);
            st4(G(S.W) + (a.its[a.n - 1] + 1) * a.wStep, ooff, cB);
        }
    }
    if (ri >= 0) {
        if constexpr (!ADJ) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if (k >= a.n) continue;
#pragma unroll
                for (int j = 0; j < K; ++j)
                    if (j == a.its[k] - a.its[0]) {
                        acc[j] += rv[k] * a.wi[k][0];
                        acc[j + 1] += rv[k] * a.wi[k][1];
                    }
            }
        }
#pragma unroll
        for (int j = 0; j < NA; ++j)
            if (j <= last) rd[ADJ ? -j : j] = acc[j];
    }
}

template <int C, unsigned MODE>
hipError_t launch_config(const StepsArgs& a, hipStream_t s, hipEvent_t e0, hipEvent_t e1)
{
    constexpr int NTH = 1024;
    constexpr StepsConfig t = kStepsConfig[C];
    auto k = k_steps<t.tz, t.tx, t.k, NTH, t.px, MODE>;
    const dim3 grid((a.ntiles * a.nshots + 7) / 8 * 8);
    if (e0 && e1) hipExtLaunchKernelGGL(k, grid, dim3(NTH), 0, s, e0, e1, 0, a);
    else hipLaunchKernelGGL(k, grid, dim3(NTH), 0, s, a);
    return hipGetLastError();
}

template <unsigned MODE>
hipError_t launch(int config, const StepsArgs& a, hipStream_t s, hipEvent_t e0, hipEvent_t e1)
{
    if (config == 0) return launch_config<0, MODE>(a, s, e0, e1);
    if (config == 1) return launch_config<1, MODE>(a, s, e0, e1);
    return launch_config<2, MODE>(a, s, e0, e1);
}

}  // namespace

hipError_t launch_steps(int config, unsigned mode, const StepsArgs& a, hipStream_t s, hipEvent_t e0, hipEvent_t e1)
{
    if (config < 0 || config >= kStepsConfigs || !wide_grid_ok(a.nz, a.nx) || a.minPad > kStepsPadMax || a.n < 1 ||
        a.n > kStepsConfig[config].k)
        return hipErrorInvalidValue;
    switch (mode) {
    case MODE_NL_FWD: return launch<MODE_NL_FWD>(config, a, s, e0, e1);
    case MODE_NL_ADJ: return launch<MODE_NL_ADJ>(config, a, s, e0, e1);
    case MODE_SRC: return launch<MODE_SRC>(config, a, s, e0, e1);
    case MODE_SRC_WIN: return launch<MODE_SRC_WIN>(config, a, s, e0, e1);
    case MODE_BORN_SCAT: return launch<MODE_BORN_SCAT>(config, a, s, e0, e1);
    case MODE_BORN_SCAT_PRE: return launch<MODE_BORN_SCAT_PRE>(config, a, s, e0, e1);
    case MODE_REC_WIN: return launch<MODE_REC_WIN>(config, a, s, e0, e1);
    case MODE_STEPS_SRC: return launch<MODE_STEPS_SRC>(config, a, s, e0, e1);
    case MODE_SRC_LAP: return launch<MODE_SRC_LAP>(config, a, s, e0, e1);
    case MODE_ADJ_GRAD: return launch<MODE_ADJ_GRAD>(config, a, s, e0, e1);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace aiso
