// Every mode and tile of k_steps on one small grid, with the threads of each
// workgroup in ascending and in descending order between its barriers: the
// slices, captures, images and traces must not depend on it.  Prints the cases
// that do.
#include <ucontext.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "steps.hip"

dim3 threadIdx, blockIdx, gridDim;

namespace fibers {

bool descending = false;
static ucontext_t scheduler;
static std::vector<ucontext_t> fiber;
static std::vector<char> ended;
static std::vector<std::vector<char>> stack;
static const std::function<void()>* body = nullptr;

static void entry()
{
    (*body)();
    ended[threadIdx.x] = 1;
    swapcontext(&fiber[threadIdx.x], &scheduler);
}

void launch(unsigned blocks, unsigned threads, const std::function<void()>& kernel)
{
    body = &kernel;
    gridDim = dim3(blocks);
    fiber.resize(threads);
    ended.resize(threads);
    stack.resize(threads, std::vector<char>(64 << 10));
    for (unsigned b = 0; b < blocks; ++b) {
        blockIdx = dim3(b);
        for (unsigned t = 0; t < threads; ++t) {
            ended[t] = 0;
            getcontext(&fiber[t]);
            fiber[t].uc_stack.ss_sp = stack[t].data();
            fiber[t].uc_stack.ss_size = stack[t].size();
            fiber[t].uc_link = nullptr;
            makecontext(&fiber[t], entry, 0);
        }
        for (unsigned left = threads; left > 0;) {
            for (unsigned i = 0; i < threads; ++i) {
                const unsigned t = descending ? threads - 1 - i : i;
                threadIdx = dim3(t);
                swapcontext(&scheduler, &fiber[t]);
                left -= ended[t];
            }
            if (left > 0 && left < threads) {
                std::printf("a barrier that not every thread reaches\n");
                std::exit(2);
            }
        }
    }
}

}  // namespace fibers

void __syncthreads()
{
    swapcontext(&fibers::fiber[threadIdx.x], &fibers::scheduler);
}

// Defined in wide.hip; the grid below satisfies it.
bool aiso::wide_grid_ok(int nz, int nx) { return (nz - 2 * FAT) % 16 == 0 && (nx - 2 * FAT) % 16 == 0; }

using namespace aiso;

namespace {

constexpr int kNz = 80 + 2 * FAT, kNx = 96 + 2 * FAT, kNts = 6, kShots = 1, kPad = 12;
constexpr long kNzx = (long)kNz * kNx;

struct Lists {
    std::vector<int> ptr;
    std::vector<int2> ent;
};

// The points (grid row and column pairs) of each tile, with `region` also
// those of its halo.
Lists lists(int config, const std::vector<int2>& points, bool region)
{
    const StepsConfig& t = kStepsConfig[config];
    const int tZ = (kNz - 2 * FAT + t.tz - 1) / t.tz, tX = (kNx - 2 * FAT + t.tx - 1) / t.tx, e = region ? FAT * (t.k - 1) : 0;
    Lists out{{0}, {}};
    for (int b = 0; b < tX; ++b)
        for (int a = 0; a < tZ; ++a) {
            for (int r = 0; r < (int)points.size(); ++r) {
                const int row = points[r].x - FAT - a * t.tz, col = points[r].y - FAT - b * t.tx;
                if (row >= -e && row < t.tz + e && col >= -e && col < t.tx + e) out.ent.push_back({steps_index(config, row, col), r});
            }
            out.ptr.push_back((int)out.ent.size());
        }
    return out;
}

// Everything two launches of a mode read and write.
struct State {
    std::vector<float> slices, W, img, dreg, sig, v2dt2, mtil, cd;
    std::vector<int2> src, rec;
};

State make_state(int nRec)
{
    std::mt19937 gen(7);
    std::normal_distribution<float> d;
    auto fill = [&](std::vector<float>& v, size_t n) { v.resize(n); for (float& x : v) x = d(gen); };
    State s;
    fill(s.slices, kShots * 4 * kNzx);
    for (long i = 0; i < (long)s.slices.size(); ++i) {              // the FAT ring is zero
        const long z = i % kNz, x = i / kNz % kNx;
        if (z < FAT || z >= kNz - FAT || x < FAT || x >= kNx - FAT) s.slices[i] = 0.f;
    }
    fill(s.W, kShots * kNts * kNzx);
    fill(s.img, kShots * kNzx);
    fill(s.mtil, kNzx);
    s.v2dt2.assign(kNzx, 0.05f);
    for (int i = 0; i < kPad; ++i) s.cd.push_back(0.9f + 0.008f * i);
    s.src = {{FAT + 30, FAT + 33}};
    for (int r = 0; r < nRec; ++r) s.rec.push_back({FAT + 31, FAT + 2 + r});
    fill(s.dreg, kShots * nRec * kNts);
    fill(s.sig, kShots * (2 * kNts));
    return s;
}

State run(int config, unsigned mode, int n, int nRec, bool descending)
{
    State s = make_state(nRec);
    const StepsConfig& t = kStepsConfig[config];
    const bool adj = mode & M_ADJ;
    const Lists src = lists(config, s.src, !adj), rec = lists(config, s.rec, adj);
    std::vector<ShotSlot> slots(kShots);
    for (int k = 0; k < kShots; ++k) {
        ShotSlot& S = slots[k];
        std::memset(&S, 0, sizeof(S));
        for (int i = 0; i < 4; ++i) S.p[i] = s.slices.data() + (4 * k + i) * kNzx;
        S.W = s.W.data() + k * kNts * kNzx;
        S.img = s.img.data() + k * kNzx;
        S.dreg = s.dreg.data() + (long)k * nRec * kNts;
        S.sig = s.sig.data() + (long)k * 2 * kNts;
        S.srcTile = S.srcOwnTile = src.ptr.data();
        S.srcEnt = S.srcOwnEnt = src.ent.data();
        S.recTile = S.recOwnTile = rec.ptr.data();
        S.recEnt = S.recOwnEnt = rec.ent.data();
    }
    StepsArgs a{};
    a.slots = slots.data();
    a.v2dt2 = s.v2dt2.data();
    a.cd = s.cd.data();
    a.mtil = s.mtil.data();
    a.nz = kNz; a.nx = kNx; a.minPad = kPad; a.nts = kNts; a.ntw = 2 * kNts; a.nshots = kShots;
    a.tilesZ = (kNz - 2 * FAT + t.tz - 1) / t.tz;
    a.ntiles = a.tilesZ * ((kNx - 2 * FAT + t.tx - 1) / t.tx);
    for (int k = 0; k < 6; ++k) a.zc[k] = a.xc[k] = 0.4f / (k + 1);
    a.wStep = kNzx;
    a.wa = 0.25f; a.wb = 0.5f; a.wc = 0.75f;
    fibers::descending = descending;
    for (int launch = 0, itw = adj ? 7 : 1; launch < 2; ++launch) {
        a.n = n;
        a.wOff = adj ? 5 * kNzx : 0;
        for (int i = 0; i < n; ++i, itw += adj ? -1 : 1) {
            a.itw[i] = itw;
            a.its[i] = itw / 2;
            a.first[i] = itw % 2 == (adj ? 1 : 0);
            a.wi[i][0] = 0.3f + i;
            a.wi[i][1] = 0.7f;
            a.fa[i] = 0.6f;
            a.fb[i] = itw % 2 ? 0.2f : 0.f;
        }
        if (launch_steps(config, mode, a, nullptr, nullptr, nullptr) != hipSuccess) {
            std::printf("mode %u was refused\n", mode);
            std::exit(2);
        }
        a.pair ^= 1;
    }
    return s;
}

bool same(const std::vector<float>& a, const std::vector<float>& b)
{
    return std::memcmp(a.data(), b.data(), a.size() * sizeof(float)) == 0;
}

}  // namespace

int main()
{
    int bad = 0;
    for (unsigned mode : {MODE_NL_FWD, MODE_NL_ADJ, MODE_SRC, MODE_SRC_WIN, MODE_BORN_SCAT, MODE_BORN_SCAT_PRE, MODE_REC_WIN,
                          MODE_STEPS_SRC, MODE_SRC_LAP, MODE_ADJ_GRAD})
        for (int config = 0; config < kStepsConfigs; ++config)
            for (int n = 1; n <= kStepsConfig[config].k; ++n)
                for (int nRec : {2, 40}) {                           // added by the computing threads, and by threads of their own
                    const State x = run(config, mode, n, nRec, false), y = run(config, mode, n, nRec, true);
                    if (same(x.slices, y.slices) && same(x.W, y.W) && same(x.img, y.img) && same(x.dreg, y.dreg) && same(x.sig, y.sig))
                        continue;
                    std::printf("mode %u, %d x %d tiles, %d steps, %d receivers: the result depends on the order of the threads\n", mode,
                                kStepsConfig[config].tz, kStepsConfig[config].tx, n, nRec);
                    ++bad;
                }
    return bad ? 1 : 0;
}
