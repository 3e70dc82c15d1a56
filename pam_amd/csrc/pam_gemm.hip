// PAM matrix products for gfx950, host side: the plan of a launch, the entry points of the C ABI for products and
// convolutions, and the scratch the library owns.  The kernel is in pam_gemm_kernel.h.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>
#include <random>

#include "pam_gemm_kernel.h"
#include "../../include/pam_hip_extra.h"
#include "../../include/pam_hip_probe.h"

using namespace pamdev;
using namespace pamgemm;

namespace {

// compute units of the current device (looked up once per device)
int cu_count()
{
    constexpr int kDevices = 64;
    static std::atomic<int> cus[kDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDevices) return 256;
    int n = cus[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        hipDeviceProp_t prop;
        n = (hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0) ? prop.multiProcessorCount : 256;
        cus[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// How a product is scheduled (see the kernel's comment on units).  bk: depth of a k-tile; kt: k-tiles per output
// tile; pieces, piece_kt: the k ranges a tile is cut into and their length in k-tiles; units = tiles x pieces.
// free: the freely shaped tiles that PAM products of operands read by 128-bit loads take instead (r = 0: none).
struct FreeShape { int r, c; };
struct Plan { int bk, kt, pieces, piece_kt; long units; FreeShape free; };

// Tuning override for experiments, per calling thread (include/pam_hip_probe.h): bk 0 = automatic (16 or 32);
// pieces 0 = automatic, > 0 that many k ranges per tile (as far as k allows).
thread_local int g_force_bk = 0, g_force_pieces = 0;

constexpr long kMostCutTiles = 8192;            // tiles of a product that cuts them (its arrival words: 64 KB)
constexpr int kResidentPerCu = 4;               // work-groups of the kernel a compute unit holds (LDS and registers)
constexpr size_t kPartBytes = (size_t)pamgemm::kPartFloats * sizeof(float);

// Wavefronts with outputs in the 64 x 64 tiles of an M x N matrix (see lane_place).
long busy_waves(long M, long N)
{
    const long full_m = M / 64, full_n = N / 64, rest_m = M % 64, rest_n = N % 64;
    return 4 * full_m * full_n + full_m * ((rest_n + 15) / 16) + full_n * ((rest_m + 15) / 16) + (std::min(rest_m, rest_n) + 15) / 16;
}

// Freely shaped tiles.  Matrices of a few tiles each whose sizes are no multiples of 64 (attention scores of 197 x 197: 16 tiles,
// 7 of them with one busy wavefront) spend work-groups on their edges, and how long a batch of them takes goes by the number
// of work-groups more than by their products.  A tile may instead have any r x c blocks of 4 x 4 outputs, one per lane, with r c up
// to 256: 25 x 10 blocks cover 197 x 197 in ten tiles, nearly without idle lanes.  c is at most 16, so that a wavefront's
// reads of the right fragment stay within 64 LDS banks (25 columns in 10 rows 34.3 us where 10 in 25 take 31.5), r at most 32.
// What a tiling costs is counted in wavefronts plus two per work-group; a freely shaped one must save a twentieth of it, as
// its own loop is up to 8 % slower (tiles of 16 x 16 blocks 10.8 us, the fixed ones 10.0), or a tenth where the fixed tiles
// are all resident (15362 x 160, k = 64, saving a seventeenth: 12.4 -> 13.2).  What takes the time is the fullest compute unit: its
// work-groups must become fewer, or the same number of fuller ones run in the slower loop (181 of 89 x 89, k = 64, three either way:
// 12.8 us, fixed tiles 12.3), and there must be more than two on it to begin with.  Where all are resident and a row of
// results is at most 32 long, the fixed tiles' wavefronts are half idle, and three such on a compute unit are as good as two full
// ones (165 of 196 x 32, k = 196: 25.7 us, fixed tiles in 32-deep k-tiles 23.3); so are four where those deeper k-tiles are taken.
// Whole tiles of 16-deep k-tiles only.
// On 2695 drawn products that the cost alone chose (attention in both directions, 16 ... 400 heads of 16 ... 400 tokens, 32 ... 128 wide; linear
// layers of 4000 ... 60000 rows; PAM products, no other mode takes these tiles): time over the fixed tiles' 0.94 where those are resident
// and 0.83 beyond, 9 and 4 % of them more than 2 % slower; with the rules on the fullest compute unit and on narrow
// results 0.91 and 0.82, 0.3 and 2.4 %; on 1108 others 0.90 and 0.83, 0.3 and 2.8 % (at worst 1.08, where a few work-groups make a second round).
// Products of 192 x 197 x 197, k = 64: 37.4 -> 31.2 us; 212 x 148 x 148, 64: 25 -> 21.4; 120 x 257 x 131, 80: 29.6 -> 25.9;
// 120 x 257 x 80, 131: 34.3 -> 22.6; 256 x 70 x 70, 64: 13.7 -> 10.7.
FreeShape free_shape(long batch, long M, long N, long K)
{
    FreeShape best{0, 0};
    const long tiles = ((M + 63) / 64) * ((N + 63) / 64), cus = cu_count(), fixed = (batch * tiles + cus - 1) / cus;
    if (batch * tiles <= 2 * cus || batch * tiles > (1L << 28) || K >= 512 || (K >= 128 && K % 32 == 0)) return best;
    const bool resident = batch * tiles <= kResidentPerCu * cus;
    if (resident && N <= 32 && (K >= 128 || fixed == 3)) return best;
    const long waves = busy_waves(M, N);
    const long fours_m = (M + 3) / 4, fours_n = (N + 3) / 4;
    long least = (waves + 2 * tiles) * (resident ? 18 : 19) / 20;
    for (long widest = std::min<long>(kFreeFoursN, fours_n); widest >= std::min<long>(6, fours_n); --widest) {
        const long tn = (fours_n + widest - 1) / widest, c = (fours_n + tn - 1) / tn, most = std::min<long>(kFreeFoursM, 256 / c), tm = (fours_m + most - 1) / most, r = (fours_m + tm - 1) / tm;
        const long cost = tm * tn * ((r * c + 63) / 64 + 2);
        if (cost < least && (batch * tm * tn + cus - 1) / cus < fixed) { least = cost; best = FreeShape{(int)r, (int)c}; }
    }
    return best;
}

constexpr int kFewRows = 4;                     // products that few_rows_kernel takes where their tiles are whole
constexpr long kFewLongest = 512;

// Products that fit the chip at once: up to 1024 tiles whose k-steps come to less than 500 per compute unit.  There a
// work-group's chain of k-tiles is what takes the time, one wavefront per SIMD issues at half rate, and cutting k much finer
// than the rule for large products does pays: pieces down to 32 k, as long as all units are resident.
bool fits_at_once(long tiles, long M, long K)
{
    return tiles <= (long)kResidentPerCu * cu_count() && tiles * K < 500L * cu_count() && !(M <= kFewRows && K <= kFewLongest);
}

// The time of a product there, in k-steps of a work-group alone on its compute unit.  A unit takes its k (0.9 of it in 32-deep
// k-tiles), 0.62 more of what is over a whole k-tile where that is the longest unit, and 280 for start, first fetch and way out; up to 1.34 times
// that where four busy work-groups share a compute unit, counted on the fullest one and on all of them about evenly, since a few full ones end
// late and the others early.  (Short pieces that end a piece-major launch do not make one fuller; any other few units over do: 644 x 864, k = 480 as 770
// units 23.6 us, as 462 of twice the length 21.0.)  Wavefronts without outputs count little, not
// nothing: they stage.  Pieces cost 13 and 3.85 each where the tile's last arriver adds them up, 45 and 0.9 each in the second kernel (20 on the
// GPU; the rest is for the host's 2.6 us of another launch, which is what a small layer's step waits for).
// One order of the sums, and so one plan, holds for a product's sizes in whatever mode: fitted on 3000 drawn products of all modes together
// (linear layers' three, dense and behind a ReLU, approximate and exact; attention's; convolutions' three, approximate and exact), each timed in both
// k-tile depths with 1 ... 64 pieces, and checked on 9565 others: 0.79 of the time of the rule below in all (products of linear layers
// 0.66 ... 0.78, convolutions' 0.75 ... 0.79, attention's 0.88 ... 0.96), 1.2 % of them more than 2 % slower, at worst 1.10.  With all units counted evenly alone, and no plan of the rule
// below among the choices, it was 0.81 and 2.6 %.
// Fullest unit: 110 of 71 x 71, k = 128 as 880 units of 64 k, four on a compute unit, 18.1 us, whole 15.8; 192 x 192, k = 12608 as 66 pieces (594 units)
// 33.3, as 57 (513) 30.8.  197 x 768, k = 192: 18.5 -> 10.2 us; beyond 500 k-steps per compute unit the two rules are even.
struct SmallTime {
    long tiles, K, cus;
    double busy;
    SmallTime(long tiles, long batch, long M, long N, long K)
        : tiles(tiles), K(K), cus(cu_count()), busy(0.13 + 0.87 * (double)(batch * busy_waves(M, N)) / (double)(4 * tiles)) {}
    double operator()(int bk, int per, int pieces) const
    {
        constexpr double kCrowd[kResidentPerCu] = {0.0, 0.01, 0.17, 0.34};
        const int n = (int)tiles * pieces;                       // (at most as many as are resident)
        const int kt = (int)((K + bk - 1) / bk), last_kt = kt - (pieces - 1) * per;
        const int counted = pieces > pamgemm::kFoldInKernel && 3 * last_kt <= per ? n - (int)tiles : n;
        const int fullest = std::max((counted + (int)cus - 1) / (int)cus, 1);
        const double even = n <= cus ? 0.0 : kCrowd[kResidentPerCu - 1] * (double)(n - cus) / (double)((kResidentPerCu - 1) * cus);
        const double step = bk == 32 ? 0.9 : 1.0, last = (double)(K - (long)(pieces - 1) * per * bk) * step + 0.62 * (double)(K & (bk - 1));
        const double unit = std::max((double)std::min((long)per * bk, K) * step, last) + (bk == 32 ? 282.0 : 280.0);
        return unit * (1.0 + busy * (0.43 * kCrowd[fullest - 1] + 0.57 * even))
            + (pieces == 1 ? 0.0 : pieces <= pamgemm::kFoldInKernel ? 12.7 + 3.85 * (double)pieces : 45.0 + 0.9 * (double)pieces);
    }
};
void small_plan(Plan& p, long tiles, long batch, long M, long N, long K)
{
    const int resident = kResidentPerCu * cu_count();
    const SmallTime small_time(tiles, batch, M, N, K);
    double best = p.units <= resident ? small_time(p.bk, p.piece_kt, p.pieces) : HUGE_VAL;
    for (int bk = 16; bk <= (K >= 128 ? 32 : 16); bk *= 2) {
        const int kt = (int)((K + bk - 1) / bk), most = (int)std::min<long>(std::max<long>((long)kt * bk / 32, 1), resident / tiles);
        for (int w = 1; w <= most; w += 1 + w / 32) {
            const int per = (kt + w - 1) / w, pieces = (kt + per - 1) / per;
            const double time = small_time(bk, per, pieces);
            if (time < best) { best = time; p.bk = bk; p.kt = kt; p.pieces = pieces; p.piece_kt = per; }
        }
    }
    p.units = tiles * p.pieces;
}

// Work-groups own 64 x 64 output tiles.  k of 128 and more in whole multiples of 32, and any k
// from 512, uses 32-deep k-tiles (fewer barriers and more bytes in flight per round, measured 3-5 %
// faster on 12608-row products), and so does ragged k of 128 and more where whole tiles are all resident
// (attention: 197); other ragged k and short k (attention: 64) 16-deep ones.
// Shapes with few output tiles and long k (dX: 12608 x 192, k = 768; dW: 192 x 768, k = 12608) cut every tile's k
// range into equal pieces, each at least 128 deep in k: few pieces by the cost model below (the tile's last
// work-group adds them up), or, where that asks for more than a work-group should add up, about two resident rounds of
// piece-major units and a second kernel.
Plan find_plan(long batch, long M, long N, long K, bool with_workspace)
{
    const long resident = (long)kResidentPerCu * cu_count();
    const long tiles = batch * ((M + 63) / 64) * ((N + 63) / 64);
    Plan p;
    p.free = FreeShape{0, 0};
    p.bk = (K >= 512 || (K >= 128 && K % 32 == 0)) ? 32 : 16;
    if (g_force_bk) p.bk = g_force_bk;
    p.kt = (int)((K + p.bk - 1) / p.bk);
    p.pieces = 1; p.piece_kt = p.kt;
    const long least = (128 + p.bk - 1) / p.bk;                       // k-tiles in 128 k
    const long most = p.kt / least;                                   // pieces a tile can be cut into
    long want = 1;
    if (g_force_pieces > 0) want = g_force_pieces;
    else if (tiles < (3 * resident) / 2 && tiles <= kMostCutTiles && with_workspace) {
        // Time of the product cut into w pieces, in k-tile times of a work-group alone on its compute unit; fitted to
        // measurements on the 12608 x 192 <-> 768 products.  A unit costs its k-tiles plus about one more (fetch of its
        // first k-tile, way out, arrival).  Up to one unit per compute unit they all run at that speed; four on a compute
        // unit each run about 1.5 times slower; beyond what is resident the rounds add up, a last round that is not
        // full costing a little more than its share.
        const long cus = resident / kResidentPerCu;
        double best = 0.0;
        for (long w = 1; w <= (most > 1 ? most : 1); ++w) {
            const long per = (p.kt + w - 1) / w, pieces = (p.kt + per - 1) / per;
            if (pieces != w) continue;                                // the same cut as a smaller w
            const long n = tiles * pieces;
            const double rounds = (double)n / (double)resident;
            const double crowd = n <= cus ? 1.0 : n <= resident ? 1.0 + 0.5 * (double)(n - cus) / (double)(resident - cus)
                                                                 : 1.5 * (rounds + 0.15 * (std::ceil(rounds) - rounds));
            const double time = (double)(per + 1) * crowd * (pieces > pamgemm::kFoldInKernel ? 1.03 : 1.0);
            if (best == 0.0 || time < best) { best = time; want = pieces; }
        }
        // More pieces than a tile's last work-group adds up itself (few tiles, very long k: the weight gradients): the
        // units are piece-major in launch order and a second kernel adds them.  Two work-groups on a compute unit issue
        // at nearly the rate of four, and a third adds little, so such a launch runs in rounds of two units per compute
        // unit: its time goes as (rounds + 0.4) x (k-tiles per piece + 1.25), the 0.4 for the skew with which a round's
        // units end, the 1.25 for a unit's start and way out.  Fitted on weight gradients of 9 ... 144 tiles with k =
        // 3152 ... 50432 (pieces of 224 k for the 192 x 768, k = 12608 one: 86 us dense, 102 us with the zeros of a
        // ReLU in the left operand; one resident round of 27 pieces, a range of them per XCD: 88 and 111 us).
        if (want > pamgemm::kFoldInKernel) {
            const long quantum = 2 * cus;
            double least_time = 0.0;
            for (long per = least;; ++per) {
                const long pieces = (p.kt + per - 1) / per;
                if (pieces <= pamgemm::kFoldInKernel) break;
                if (pieces > most) continue;
                const long n = tiles * pieces;
                long rounds = (n - n / 50 + quantum - 1) / quantum;               // (2 % over whole rounds still counts as those)
                if (rounds < 1) rounds = 1;
                const double time = ((double)rounds + 0.4) * ((double)per + 1.25);
                if (least_time == 0.0 || time < least_time) { least_time = time; want = pieces; }
            }
        }
    }
    if (want > (g_force_pieces > 0 ? (long)p.kt : most)) want = g_force_pieces > 0 ? (long)p.kt : most;
    if (with_workspace && want > 1 && tiles <= kMostCutTiles) {
        p.piece_kt = (int)((p.kt + want - 1) / want);
        p.pieces = (p.kt + p.piece_kt - 1) / p.piece_kt;
    }
    p.units = tiles * p.pieces;
    // whole tiles of ragged k, all resident: 32-deep k-tiles (192 of 197 x 64, k = 197 29.7 -> 29.0 us and 31.4 -> 30.5 with operands along k;
    // 13642 x 233, 364 58.5 -> 57.0, its gradients 1 to 3 %; with a ReLU's zeros 29.7 -> 26.6)
    if (p.pieces == 1 && p.bk == 16 && K >= 128 && p.units <= resident && !g_force_bk) { p.bk = 32; p.kt = p.piece_kt = (int)((K + 31) / 32); }
    if (with_workspace && g_force_bk == 0 && g_force_pieces == 0 && fits_at_once(tiles, M, K)) small_plan(p, tiles, batch, M, N, K);
    return p;
}

// The plans of a thread's last products by their sizes: a call asks for its plan twice (scratch, launch), and a program for the
// same ones again and again.  (Finding one takes up to 2 us, and 5 for one tile of very long k.)
Plan make_plan(long batch, long M, long N, long K, bool with_workspace)
{
    const auto find = [&] {
        Plan p = find_plan(batch, M, N, K, with_workspace);
        if (p.pieces == 1 && !g_force_bk && !g_force_pieces) p.free = free_shape(batch, M, N, K);
        return p;
    };
    if (g_force_bk || g_force_pieces) return find();
    struct Found { long batch, M, N, K; int cus; bool with_workspace; Plan plan; };
    constexpr int kFound = 256;                    // (eight bits; 22 KB)
    thread_local Found found[kFound] = {};
    const int cus = cu_count();
    // (the top bits of a sum of products with odd 64-bit numbers: most sizes are multiples of 32, and a sum of small multiples put
    // the three products of a layer of such sizes in one place)
    const uint64_t mixed = (uint64_t)batch * 0x9e3779b97f4a7c15u + (uint64_t)M * 0xc2b2ae3d27d4eb4fu + (uint64_t)N * 0x165667b19e3779f9u
        + (uint64_t)K * 0xd6e8feb86659fd93u + (with_workspace ? 0xa0761d6478bd642fu : 0u);
    Found& f = found[((mixed ^ (mixed >> 32)) * 0x9e3779b97f4a7c15u) >> 56];
    if (f.batch != batch || f.M != M || f.N != N || f.K != K || f.cus != cus || f.with_workspace != with_workspace)
        f = Found{batch, M, N, K, cus, with_workspace, find()};
    return f.plan;
}

// Whether a launch's work-groups lower their priority by quarters of their k-tiles, so that those on a compute unit end
// together instead of one after the other.  What matters is how much of the chip the last round leaves idle.  Where it
// fills more than half of it the steps gain 3 to 14 % (in the first round or two, less the more rounds there are); where it
// has at most one work-group per compute unit they lose 2 to 11 %: units that would have ended apart and let the rest
// begin early all end at once, and the rest runs alone (on 1024 resident ones: 1328 work-groups 0.97 of the time
// without steps where the tiles are whole, 1088 1.08, 2304 1.04, 2049 1.05, 2048 0.95, 1024 0.93, 640 0.88, 512 and less 1.00 to
// 1.03).  Between the two, in the second and third round, they gain 2 to 3 % in units of twenty and more k-tiles, and in
// shorter ones that are whole tiles of whole 64 x 64 outputs; elsewhere between -4 and +6 %.  In a launch of several
// rounds each step must cover more than one k-tile of its unit: units of four or five k-tiles lose 2 to 6 % there, and of the
// exact gradients', with three operations per product, those of up to seven in the third round and up to nine beyond, 2 to 10 %.
// On 4151 products of drawn shapes, geometric mean of the time over that without steps: always 0.989, this rule 0.980, the
// better of the two each time 0.979.
// (Freely shaped tiles take the steps in a mostly full second round at any depth: 192 products of 197 x 197, k = 64 in 1920
// work-groups 34.3 -> 33.1 us, 217 of 197 x 159 29.0 -> 27.1.)
bool priority_steps(const Plan& p, long M, long N, bool exact)
{
    const long cus = cu_count(), resident = (long)kResidentPerCu * cus;
    if (p.units <= resident) return p.units > resident / 2;
    // (piece-major launches end with the tiles' last pieces, which may be short: a few of at most a third of the length behind
    // full rounds do not count, 2052 units of 224 k of which the last 36 have 64: 0.95; from half the length on they do, 1.02 to 1.10)
    const long tiles = p.units / p.pieces, extra = p.units % resident, tail = p.kt - (long)(p.pieces - 1) * p.piece_kt;
    const long counted = p.pieces > pamgemm::kFoldInKernel && extra <= tiles && 3 * tail <= p.piece_kt ? p.units - extra : p.units;
    const long rounds = (counted + resident - 1) / resident, last = (counted - 1) % resident + 1;
    const bool most = last > resident / 2;
    if (p.free.r > 0 && most && rounds <= 2) return true;
    if (p.piece_kt < (!exact || (most && rounds <= 2) ? 6 : most && rounds <= 3 ? 8 : 10)) return false;
    return most || (last > cus && rounds <= 3 && (p.piece_kt >= 20 || (p.pieces == 1 && M % 64 == 0 && N % 64 == 0)));
}

// What a launch makes of its sizes' plan.  conv: the right operand is an image's patches; quads: both operands are read by
// 128-bit loads.
Plan launch_plan(Plan p, bool pam, bool conv, bool quads, long batch, long M, long N, long K)
{
    // (convolutions stay with 16-deep k-tiles for ragged k of whole tiles: half a k-tile left over costs them more, 100 images of
    // 16 x 32 x 32 to 64 channels, k = 144: 59.9 us, in 32-deep ones 64.7)
    if (conv && p.pieces == 1 && p.bk == 32 && K < 512 && K % 32 != 0 && !g_force_bk) { p.bk = 16; p.kt = p.piece_kt = (int)((K + 15) / 16); }
    if (!pam || conv || !quads) p.free = FreeShape{0, 0};
    if (p.free.r > 0) {
        p.bk = 16; p.kt = p.piece_kt = (int)((K + 15) / 16);
        p.units = batch * ((M + 4 * p.free.r - 1) / (4 * p.free.r)) * ((N + 4 * p.free.c - 1) / (4 * p.free.c));
    }
    return p;
}

// workspace of a plan that cuts tiles: [arrival words, one per tile][one piece per unit].  The words' part has one size
// for every shape, so that products of different shapes that share a workspace never write pieces over each other's
// words (a word that does not carry the launch's tag costs its first arriver two more round trips).
constexpr size_t kArriveBytes = (size_t)kMostCutTiles * sizeof(unsigned long long);
struct Space { size_t partial, total; };
Space plan_space(const Plan& p)
{
    Space w{0, 0};
    if (p.pieces > 1) {
        w.partial = kArriveBytes;
        w.total = w.partial + (size_t)p.units * kPartBytes;
    }
    return w;
}

// Tags of the launches that cut tiles: a 40-bit counter that starts at a random value.
unsigned long long next_tag()
{
    static std::atomic<unsigned long long> counter{[] {
        std::random_device rd;
        return ((unsigned long long)rd() << 32) | rd();
    }()};
    return counter.fetch_add(1, std::memory_order_relaxed) & pamgemm::kTagMask;
}

// sums over nothing: +0, plus the bias
__global__ __launch_bounds__(256) void empty_k_kernel(float* __restrict__ y, long y_sb, long y_sr, long y_sc, long batch, int M, int N,
                                                     const float* __restrict__ bias)
{
    const long per = (long)M * N, idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= batch * per) return;
    const long b = idx / per, rem = idx % per;
    y[b * y_sb + (rem / N) * y_sr + (rem % N) * y_sc] = bias ? 0.0f + bias[rem % N] : 0.0f;
}

// Cut tiles of many pieces: the pieces of every tile added in ascending order from +0 by a kernel of its own, one
// lane per 128-bit row of the tile (work-groups of 128 lanes, eight per tile); eight pieces' loads in flight.
__global__ __launch_bounds__(128) void fold_kernel(pamgemm::GemmArgs g)
{
    using pamgemm::v4f;
    const int flat = blockIdx.x / 8, i = (blockIdx.x % 8) / 2, tid = (blockIdx.x % 2) * 128 + threadIdx.x;
    v4f total = {0.0f, 0.0f, 0.0f, 0.0f};
    const long first = (long)flat * g.pieces;
    int p = 0;
    for (; p + 8 <= g.pieces; p += 8) {
        v4f v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = *pamgemm::piece_row(g.partial, first + p + c, i, tid);
#pragma unroll
        for (int c = 0; c < 8; ++c) total += v[c];
    }
    for (; p < g.pieces; ++p) total += *pamgemm::piece_row(g.partial, first + p, i, tid);
    const int zb = flat / g.tiles, tile = flat - zb * g.tiles, tr = tile / g.ntn;
    const int row0 = tr * 64, col0 = (tile - tr * g.ntn) * 64;
    const pamgemm::LanePlace place = pamgemm::lane_place(tid, row0, col0, g.M, g.N);
    const int r = row0 + place.ty * 4 + i, c = col0 + place.tx * 4;
    if (r >= g.M) return;
    float* dst = g.Y + (long)zb * g.y_sb + (long)r * g.y_sr + (long)c * g.y_sc;
    const float sums[4] = {total.x, total.y, total.z, total.w};
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (c + j < g.N) dst[(long)j * g.y_sc] = g.bias ? sums[j] + g.bias[c + j] : sums[j];
}

// Products of at most kFewRows rows and short sums (one decoding step of attention: a query against the keys and values of
// every head).  The matrix kernel's 64 x 64 tiles leave 60 or more of 64 rows empty there and run a k-tile at a time, each a
// round trip to memory; here a work-group takes 64 columns of one matrix, a k-tile is 64 deep with all of a lane's loads in flight and the
// next tile's loads run under the sums of this one.  Wavefront r sums row r, one column per lane, k ascending from +0: the
// order of whole tiles.  Bound by the latency of two to three rounds of loads.  256 products of 1 x 120, k = 64: 8.6 -> 4.4 us,
// of 1 x 64, k = 120: 13.8 -> 5.9; 512 of 4 x 512, k = 64: 35 -> 18; 1600 of 4 x 64, k = 512: 90 -> 49.
// Zeros (masked keys, padded caches, activations behind a ReLU) contribute nothing: where a tile's only values outside the
// plain window are zeros, a product is selected away by one test of both operands, since no sum that starts from +0 becomes -0.
// (The general definition for such tiles was up to 45 % slower than the matrix kernel with its paths for zeros: 256 of 1 x 120,
// k = 64, a third of the right operand zeros 12.2 us, matrix kernel 10.2, now 5.3; 1600 of 4 x 64, k = 512 156, 121, 74.)
// Other values outside the window (subnormal, infinite, huge, tiny) take the general definition: 100 us at the latter, 207
// in the matrix kernel.  With up to four rows this kernel was the faster one in every class of values at eleven shapes, 1.6 to
// 4 times.  A plan that cuts k (k of 256 and more on fewer than 1536 tiles) goes to the matrix kernel, whose pieces the
// sums follow; beyond kFewLongest nothing was measured.
constexpr int kFewDepth = 64;
template <bool ALONG_K>                   // which index of the right operand is contiguous (or nearer to it)
__global__ __launch_bounds__(256) void few_rows_kernel(pamgemm::GemmArgs g)
{
    using namespace pamgemm;
    constexpr int kEach = kFewDepth * 64 / 256, kPitch = 64 + 1;
    enum { kPlain = 0, kZeros = 1, kOdd = 2 };
    __shared__ uint32_t right[kFewDepth * kPitch];
    __shared__ __attribute__((aligned(16))) uint32_t left[kFewRows][kFewDepth];
    __shared__ int classes[kFewRows];
    const int zb = blockIdx.x / g.ntn, col0 = (blockIdx.x - zb * g.ntn) * 64;
    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const float* lbase = g.L.p + (long)zb * g.L.sb + (long)min(wave, g.M - 1) * g.L.sr;
    const float* rbase = g.R.p + (long)zb * g.R.sb;
    uint32_t rv[kEach], lv;
    // (indexes past the end repeat the last one: their values are not summed)
    auto load = [&](int k0) __attribute__((always_inline)) {
        lv = f2u(lbase[(long)min(k0 + lane, g.K - 1) * g.L.sk]);
#pragma unroll
        for (int i = 0; i < kEach; ++i) {
            const int k = ALONG_K ? lane : wave + 4 * i, n = ALONG_K ? wave + 4 * i : lane;
            rv[i] = f2u(rbase[(long)min(col0 + n, g.N - 1) * g.R.sr + (long)min(k0 + k, g.K - 1) * g.R.sk]);
        }
    };
    float acc = 0.0f;
    load(0);
    for (int k0 = 0; k0 < g.K; k0 += kFewDepth) {
        uint32_t seen = window(lv);
#pragma unroll
        for (int i = 0; i < kEach; ++i) {
            const int k = ALONG_K ? lane : wave + 4 * i, n = ALONG_K ? wave + 4 * i : lane;
            right[k * kPitch + n] = rv[i];
            seen = max(seen, window(rv[i]));
        }
        left[wave][lane] = lv;
        int mine = kPlain;
        if (__ballot(seen >= kWindowSpan) != 0ull) {
            uint32_t odd = (lv << 1) != 0u ? window(lv) : 0u;
#pragma unroll
            for (int i = 0; i < kEach; ++i) odd = max(odd, (rv[i] << 1) != 0u ? window(rv[i]) : 0u);
            mine = __ballot(odd >= kWindowSpan) != 0ull ? kOdd : kZeros;
        }
        if (lane == 0) classes[wave] = mine;
        __syncthreads();
        const int cls = max(max(classes[0], classes[1]), max(classes[2], classes[3]));
        const int depth = min(kFewDepth, g.K - k0);
        if (k0 + kFewDepth < g.K) load(k0 + kFewDepth);
        if (wave < g.M) {
            const uint32_t* lrow = left[wave];
            if (cls == kPlain) {
#pragma unroll 16
                for (int k = 0; k < depth; ++k) acc = acc + u2f(lrow[k] + (right[k * kPitch + lane] - kBias));
            } else if (cls == kZeros) {
#pragma unroll 16
                for (int k = 0; k < depth; ++k) {
                    const uint32_t l = lrow[k], r = right[k * kPitch + lane];
                    acc = acc + (min(l << 1, r << 1) != 0u ? u2f(l + (r - kBias)) : 0.0f);
                }
            } else {
#pragma unroll 4
                for (int k = 0; k < depth; ++k) acc = acc + pam_mul(u2f(lrow[k]), u2f(right[k * kPitch + lane]));
            }
        }
        __syncthreads();
    }
    const int c = col0 + lane;
    if (wave < g.M && c < g.N)
        g.Y[(long)zb * g.y_sb + (long)wave * g.y_sr + (long)c * g.y_sc] = g.bias ? acc + g.bias[c] : acc;
}

int load_kind(long s_row, long s_k, long s_batch, const float* p, long rows, long K)
{
    bool aligned = ((reinterpret_cast<uintptr_t>(p) & 15u) == 0) && (s_batch % 4 == 0);
    if (s_k == 1 && aligned && s_row % 4 == 0 && K % 4 == 0 && K >= 4) return LOAD_KVEC;
    if (s_row == 1 && aligned && s_k % 4 == 0 && rows % 4 == 0 && rows >= 4) return LOAD_RVEC;
    return LOAD_ANY;
}

// Two operands that are both contiguous one way or the other, if not in aligned lines of whole quads, are read by 128-bit
// loads all the same (where one of them has other strides, the loader value by value stays).  Value by value, with 64-bit
// addresses: products 3149 x 103 x 951 24.9 / 31.7 / 27.7 us, now 20.6 / 26.5 / 25.4; 192 of 197 x 64, k = 197 31.7, now 29.0;
// 13642 x 364 x 233: 66.3 / 71.5, now 61.4 / 66.8.  Aligned operands keep instances of their own: with the tests for a line's end
// in them, products of a few k-tiles ran 1 to 4 % slower.
int odd_kind(int kind) { return kind == LOAD_KVEC ? LOAD_KODD : kind == LOAD_RVEC ? LOAD_RODD : kind; }
void odd_lines(long l_row, long l_k, long M, long r_row, long r_k, long N, long K, int& lk, int& rk)
{
    if (lk != LOAD_ANY && rk != LOAD_ANY) return;
    auto contiguous = [&](long s_row, long s_k, long rows) { return s_k == 1 && K >= 4 ? LOAD_KODD : s_row == 1 && rows >= 4 ? LOAD_RODD : LOAD_ANY; };
    const int l = lk != LOAD_ANY ? odd_kind(lk) : contiguous(l_row, l_k, M), r = rk != LOAD_ANY ? odd_kind(rk) : contiguous(r_row, r_k, N);
    if (l != LOAD_ANY && r != LOAD_ANY) { lk = l; rk = r; }
}

// One contiguous range of units per XCD (see the kernel), rounded up to whole work-groups per XCD; returns the work-groups.
unsigned spread_over_xcds(GemmArgs& g)
{
    g.xcd_chunk = (g.units + XCDS - 1) / XCDS;
    return (unsigned)(g.xcd_chunk * XCDS);
}

template <int MODE>
void launch_mode(const Plan& p, int lk, int rk, hipStream_t st, const GemmArgs& g)
{
    // Piece-major launches keep the launch order: all XCDs then work on the same few k ranges at a time (each L2 fetches them,
    // from the memory-side cache), where ranges would have every L2 hold three or four k ranges of both operands at
    // once -- measured 3 % (dense) to 9 % (left operand with zeros) slower.
    GemmArgs ga = g;
    unsigned groups = (unsigned)p.units;
    if (p.units >= 64 && (p.pieces == 1 || g.fold_here)) groups = spread_over_xcds(ga);
    if (p.bk == 32) pamgemm::launch_gemm<32, MODE>(lk, rk, groups, st, ga);
    else pamgemm::launch_gemm<16, MODE>(lk, rk, groups, st, ga);
}

int gemm(const char* what, int mode, long batch, long M, long N, long K,
         const float* l, long l_sb, long l_sr, long l_sc, const float* r, long r_sb, long r_sr, long r_sc,
         const float* d, long d_sb, long d_sr, long d_sc, float* y, long y_sb, long y_sr, long y_sc,
         float offset, void* workspace, size_t workspace_bytes, void* stream, const ConvGeom* conv = nullptr,
         const float* bias = nullptr)
{
    if (batch < 0 || M < 0 || N < 0 || K < 0) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: negative size", what);
    if (batch == 0 || M == 0 || N == 0) return PAM_HIP_OK;
    // with K == 0 the operands are empty (and may be null): the sums over nothing are +0 (plus the bias)
    if (((!l || !r) && K > 0) || !y || (mode >= MODE_BWD_DL && !d)) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: null pointer", what);
    if (M > (1L << 30) || N > (1L << 30) || K > (1L << 30) || batch > (1L << 30) || batch * ((M + 63) / 64) * ((N + 63) / 64) > 0x7fffff00L)
        return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: dimension too large (sizes and batch <= 2^30, output tiles of all matrices < 2^31)", what);
    hipStream_t st = (hipStream_t)stream;

    if (K == 0) {                                  // (the operands are empty, and may be null)
        const long n = batch * M * N;
        hipLaunchKernelGGL(empty_k_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, y, y_sb, y_sr, y_sc, batch, (int)M, (int)N, bias);
        return pamhost::check_launch(what);
    }
    const bool usable = workspace != nullptr && (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0;
    Plan p = make_plan(batch, M, N, K, usable);
    if (p.pieces > 1 && plan_space(p).total > workspace_bytes) p = make_plan(batch, M, N, K, false);       // whole tiles
    int lk = load_kind(l_sr, l_sc, l_sb, l, M, K);
    int rk = conv ? LOAD_CONV : load_kind(r_sc, r_sr, r_sb, r, N, K);
    if (!conv && mode != MODE_STD) odd_lines(l_sr, l_sc, M, r_sc, r_sr, N, K, lk, rk);
    if (conv && conv->quads && !conv->transposed && mode == MODE_PAM && lk == LOAD_KVEC && K % 4 == 0 && (reinterpret_cast<uintptr_t>(r) & 15u) == 0 && r_sb % 4 == 0)
        rk = LOAD_CONVQ;
    else if (conv && conv->row_quads && !conv->transposed && mode != MODE_STD && lk == LOAD_KVEC && N % 4 == 0)
        rk = LOAD_CONVR;
    else if (conv && conv->row_quads && conv->transposed && mode != MODE_STD && lk == LOAD_KVEC && K % 4 == 0)
        rk = LOAD_CONVK;
    const bool few = mode == MODE_PAM && !conv && M <= kFewRows && K <= kFewLongest && p.pieces == 1 && offset == 1.0f && g_force_bk == 0 && g_force_pieces == 0;
    p = launch_plan(p, mode == MODE_PAM && !few, conv != nullptr, lk != LOAD_ANY && rk != LOAD_ANY, batch, M, N, K);
    const Space sp = plan_space(p);

    GemmArgs g;
    g.L = Operand{l, l_sb, l_sr, l_sc};
    g.R = Operand{r, r_sb, r_sc, r_sr};            // R's "row" index is the output column
    g.D = d; g.d_sb = d_sb; g.d_sr = d_sr; g.d_sc = d_sc;
    g.Y = y; g.y_sb = y_sb; g.y_sr = y_sr; g.y_sc = y_sc;
    g.bias = bias;
    g.M = (int)M; g.N = (int)N; g.K = (int)K;
    const long tile_m = p.free.r > 0 ? 4 * p.free.r : 64, tile_n = p.free.r > 0 ? 4 * p.free.c : 64;
    g.ntn = (int)((N + tile_n - 1) / tile_n); g.tiles = (int)(((M + tile_m - 1) / tile_m) * g.ntn);
    g.free_r = p.free.r; g.free_c = p.free.c;
    g.pieces = p.pieces; g.piece_kt = p.piece_kt; g.units = (int)p.units;
    g.xcd_chunk = 0;
    g.steps = priority_steps(p, M, N, mode >= MODE_BWD_DL) ? 1 : 0;
    g.fold_here = p.pieces > 1 && p.pieces <= pamgemm::kFoldInKernel;
    g.arrive = p.pieces > 1 ? (unsigned long long*)workspace : nullptr;
    g.tag = g.fold_here ? next_tag() : 0;
    g.partial = p.pieces > 1 ? (float*)((char*)workspace + sp.partial) : nullptr;
    g.off = offset; g.off_add = 0; g.has_off = 0;
    if (mode != MODE_STD && offset != 1.0f) {
        uint32_t bits; memcpy(&bits, &offset, sizeof bits);
        g.has_off = std::isnormal(offset) ? 1 : 2;
        g.off_add = bits - kBias;
    }

    g.cv = conv ? *conv : ConvGeom{nullptr, nullptr, 0, 0, 0, 0, 0};

    if (few) {
        const unsigned groups = (unsigned)(batch * g.ntn);
        if (g.R.sk <= g.R.sr) hipLaunchKernelGGL(few_rows_kernel<true>, dim3(groups), dim3(256), 0, st, g);
        else hipLaunchKernelGGL(few_rows_kernel<false>, dim3(groups), dim3(256), 0, st, g);
        return pamhost::check_launch(what);
    }
    if (p.free.r > 0) {
        const unsigned groups = spread_over_xcds(g);
        launch_free(odd_kind(lk), odd_kind(rk), groups, st, g);
        return pamhost::check_launch(what);
    }
    switch (mode) {
    case MODE_PAM: launch_mode<MODE_PAM>(p, lk, rk, st, g); break;
    case MODE_STD: launch_mode<MODE_STD>(p, lk, rk, st, g); break;
    case MODE_BWD_DL: launch_mode<MODE_BWD_DL>(p, lk, rk, st, g); break;
    default: launch_mode<MODE_BWD_DR>(p, lk, rk, st, g); break;
    }
    if (p.pieces > 1 && !g.fold_here)
        hipLaunchKernelGGL(fold_kernel, dim3((unsigned)(p.units / p.pieces * 8)), dim3(128), 0, st, g);
    return pamhost::check_launch(what);
}

// ---------------------------------------------------------------- convolution as a product with image patches
// groups: channels and filters fall into `g` groups that do not mix (weights [co][c / g][kh][kw]); K() is the
// length of one group's sums
struct ConvShape {
    long batch, c, h, w, co, kh, kw, sh, sw, ph, pw, ho, wo, g;
    long cg() const { return c / g; } long cog() const { return co / g; }
    long K() const { return cg() * kh * kw; } long L() const { return ho * wo; }
};

__global__ __launch_bounds__(256) void conv_tables_kernel(int2* __restrict__ ktab, int2* __restrict__ ltab, int K, int L,
                                                         int kh, int kw, int H, int W, int wo, int sh, int sw, int ph, int pw)
{
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx < K) {
        const int c = idx / (kh * kw), rem = idx % (kh * kw), i = rem / kw, j = rem % kw;
        ktab[idx] = make_int2(c * H * W + i * W + j, (i << 16) | j);
    }
    if (idx < L) {
        const int h0 = (idx / wo) * sh - ph, w0 = (idx % wo) * sw - pw;
        ltab[idx] = make_int2(h0 * W + w0, (int)(((unsigned)h0 << 16) | ((unsigned)w0 & 0xffffu)));
    }
}

// out = `copies` copies of in[0 .. n), each value (*) off if has_off
__global__ __launch_bounds__(256) void scale_kernel(const float* __restrict__ in, float* __restrict__ out, size_t n, size_t copies, float off,
                                                    int has_off)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n * copies; i += (size_t)gridDim.x * 256) {
        const float v = in[i % n];
        out[i] = has_off ? pam_mul(v, off) : v;
    }
}
void launch_scale(const float* in, float* out, size_t n, size_t copies, float off, bool has_off, hipStream_t st)
{
    size_t blocks = (n * copies + 1023) / 1024;
    if (blocks > (1u << 20)) blocks = 1u << 20;
    hipLaunchKernelGGL(scale_kernel, dim3((unsigned)blocks), dim3(256), 0, st, in, out, n, copies, off, has_off ? 1 : 0);
}

// wf[c][co][i][j] = w[co][c][kh-1-i][kw-1-j] (*) off: the weights of the convolution over the
// upstream gradient that yields the gradient of the input (stride 1)
// (with groups: c runs over all channels, co over the filters of c's group, and w is [filters][c per group][kh][kw])
// (`copies` of them one after the other: see kReplicateBytes)
__global__ __launch_bounds__(256) void flip_weights_kernel(const float* __restrict__ w, float* __restrict__ wf, int c, int cog, int cg, int kh, int kw,
                                                          float off, int has_off, int copies)
{
    const long at = (long)blockIdx.x * 256 + threadIdx.x, n = (long)c * cog * kh * kw;
    if (at >= n * copies) return;
    const int idx = (int)(at % n);
    const int j = idx % kw, i = (idx / kw) % kh, o = (idx / (kw * kh)) % cog, ci = idx / (kw * kh * cog);
    const int filter = (ci / cg) * cog + o;
    const float v = w[(((long)filter * cg + ci % cg) * kh + (kh - 1 - i)) * kw + (kw - 1 - j)];
    wf[at] = has_off ? pam_mul(v, off) : v;
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

int conv_shape(const char* what, ConvShape& s)
{
    if (s.batch < 0 || s.c <= 0 || s.h <= 0 || s.w <= 0 || s.co <= 0 || s.kh <= 0 || s.kw <= 0 || s.sh <= 0 || s.sw <= 0 || s.ph < 0 || s.pw < 0)
        return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: bad geometry", what);
    if (s.g <= 0 || s.c % s.g != 0 || s.co % s.g != 0 || s.g > 65535)
        return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: groups must divide the channel and filter counts", what);
    s.ho = (s.h + 2 * s.ph - s.kh) / s.sh + 1;             // (in + 2 pad - (k - 1) - 1) / stride + 1 (pam/pam_ops.py:137-138)
    s.wo = (s.w + 2 * s.pw - s.kw) / s.sw + 1;
    if (s.h + 2 * s.ph < s.kh || s.w + 2 * s.pw < s.kw) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: kernel larger than the padded image", what);
    if (s.c * s.h * s.w >= (1L << 31) || s.h >= 32768 || s.w >= 32768 || s.kh >= 32768 || s.kw >= 32768 || s.ph >= 16384 || s.pw >= 16384)
        return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: image too large for the patch tables", what);
    return PAM_HIP_OK;
}

// A grouped convolution is one launch over (image, group) pairs: unit z = image * groups + group finds its rows of the
// image, of the upstream gradient and of the output at z times one group's size, since an image's groups lie one after
// the other.  Only the weights do not follow that pattern (every image uses all of them), so where a product reads them
// it gets one copy per image -- up to this many bytes of copies; beyond, the groups are launched one by one.
constexpr size_t kReplicateBytes = 32u << 20;
bool replicated(const ConvShape& s) { return s.g > 1 && (size_t)s.batch * s.co * s.K() * sizeof(float) <= kReplicateBytes; }

// workspace: [k table][l table][operand scaled by the offset, or the weights' copies, if any][split-k partial tiles]
// which: 0 forward, 1 weight gradient approximate, 2 weight gradient exact
struct ConvSpace { size_t tables, scaled, total; };
ConvSpace conv_space(const ConvShape& s, int which, bool has_off)
{
    ConvSpace w;
    w.tables = align256((size_t)(s.K() + s.L()) * sizeof(int2));
    const size_t copies = replicated(s) ? (size_t)s.batch : 1;
    size_t scaled_elems = 0;
    if (which == 0) scaled_elems = (has_off || copies > 1) ? copies * s.co * s.K() : 0;
    else if (which == 1) scaled_elems = has_off ? (size_t)s.batch * s.co * s.L() : 0;
    else scaled_elems = copies > 1 ? copies * s.co * s.K() : 0;
    w.scaled = align256(scaled_elems * sizeof(float));
    const long launches = s.g > 1 && (which == 1 || replicated(s)) ? s.batch * s.g : s.batch;
    size_t split = which != 0 ? pam_hip_gemm_workspace_bytes(launches, s.cog(), s.K(), s.L())
                              : pam_hip_gemm_workspace_bytes(launches, s.cog(), s.L(), s.K());
    w.total = w.tables + w.scaled + split;
    return w;
}

int conv_prepare(const char* what, const ConvShape& s, const ConvSpace& sp, void* workspace, size_t workspace_bytes,
                 hipStream_t st, ConvGeom& cv, bool transposed)
{
    if (!workspace || workspace_bytes < sp.total)
        return pamhost::fail(PAM_HIP_ERR_WORKSPACE, "%s: workspace of %zu bytes needed", what, sp.total);
    int2* ktab = (int2*)workspace; int2* ltab = ktab + s.K();
    const long n = s.K() > s.L() ? s.K() : s.L();
    hipLaunchKernelGGL(conv_tables_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, ktab, ltab, (int)s.K(), (int)s.L(),
                       (int)s.kh, (int)s.kw, (int)s.h, (int)s.w, (int)s.wo, (int)s.sh, (int)s.sw, (int)s.ph, (int)s.pw);
    const bool quads = s.ph == 0 && s.pw == 0 && s.kw % 4 == 0 && s.w % 4 == 0 && s.sw % 4 == 0;
    const bool row_quads = s.sw == 1 && s.wo % 4 == 0 && s.w >= 4;
    cv = ConvGeom{ktab, ltab, (int)s.h, (int)s.w, transposed ? 1 : 0, quads ? 1 : 0, row_quads ? 1 : 0};
    return PAM_HIP_OK;
}

// The gradient of the input of a stride-1 convolution is itself a convolution: of the upstream
// gradient [co, ho, wo], padded by (k - 1 - pad), with the weights flipped and their two channel
// indices exchanged.  `t` is that convolution's geometry (its "image" is the upstream gradient).
int input_gradient_shape(const char* what, const ConvShape& s, ConvShape& t)
{
    if (s.sh != 1 || s.sw != 1) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: the input gradient in place needs stride 1", what);
    if (s.ph > s.kh - 1 || s.pw > s.kw - 1) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: padding larger than kernel - 1", what);
    t = ConvShape{s.batch, s.co, s.ho, s.wo, s.c, s.kh, s.kw, 1, 1, s.kh - 1 - s.ph, s.kw - 1 - s.pw, 0, 0, s.g};
    int rc = conv_shape(what, t);
    if (rc != PAM_HIP_OK) return rc;
    if (t.ho != s.h || t.wo != s.w) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: geometry does not invert", what);
    return PAM_HIP_OK;
}

// workspace: [k table][l table][flipped weights][split-k partial tiles]
ConvSpace input_gradient_space(const ConvShape& t)
{
    ConvSpace w;
    w.tables = align256((size_t)(t.K() + t.L()) * sizeof(int2));
    const bool copies = replicated(t);
    w.scaled = align256((copies ? (size_t)t.batch : 1) * t.co * t.K() * sizeof(float));
    w.total = w.tables + w.scaled + pam_hip_gemm_workspace_bytes(copies ? t.batch * t.g : t.batch, t.cog(), t.L(), t.K());
    return w;
}

// ---------------------------------------------------------------- convolutions with small groups (depthwise among them)
// A group of a few channels and filters is a handful of terms per output ((c / groups) kh kw of them) and fills a few rows
// of a matrix tile; these kernels compute such convolutions directly, in the order the matrix kernel would: terms in
// ascending k from +0, a padding position contributing the product with +0.
// gin / gout: channels of a group that a sum runs over / that it produces.
struct DirectGeom { int IC, H, W, ho, wo, kh, kw, sh, sw, ph, pw, gin, gout; };

// out[b][p][oh][ow], p = g gout + oc, = sum over q < gin and (i, j) of term(weight, img[b][g gin + q][oh sh - ph + i][ow sw - pw + j]).
// The weight: w[p][q][i][j], or with `transposed` w[g gin + q][oc][kh - 1 - i][kw - 1 - j] (the input gradient: img = the
// upstream gradient, the stride-1 geometry of that convolution, the sum over a group's filters).
// EXACT false: term = (weight (*) off) (*) v -- the forward and the approximate input gradient; EXACT true:
// term = pam_bwd(d, weight, v) with the offset on the weight, d = the output position's own forward input.
// SIDE: the kernel is SIDE x SIDE taps and the loops over them are unrolled (all of a channel's loads in flight
// together); 0: any kernel size.
template <bool EXACT, int SIDE>
__global__ __launch_bounds__(256) void direct_conv_kernel(const float* __restrict__ img, const float* __restrict__ w, const float* __restrict__ d,
                                                         float* __restrict__ out, long total, int planes, DirectGeom q, int transposed, float off,
                                                         int has_off)
{
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    int ow, oh, p; long b;                                                // idx = ((b planes + p) ho + oh) wo + ow
    if (total <= 0x7fffffffL) {                                           // (32-bit divisions where they do: the 64-bit ones are long)
        const int at = (int)idx, hw = q.wo * q.ho, plane = at / hw, l = at - plane * hw, b32 = plane / planes;
        oh = l / q.wo; ow = l - oh * q.wo; p = plane - b32 * planes; b = b32;
    } else {
        const long plane = idx / ((long)q.wo * q.ho);
        ow = (int)(idx % q.wo); oh = (int)((idx / q.wo) % q.ho); p = (int)(plane % planes); b = plane / planes;
    }
    const int kh = SIDE ? SIDE : q.kh, kw = SIDE ? SIDE : q.kw;
    const int g = p / q.gout, oc = p % q.gout, taps = kh * kw;
    const float dv = EXACT ? d[idx] : 0.0f;
    float acc = 0.0f;
    for (int c = 0; c < q.gin; ++c) {
        const float* base = img + (b * q.IC + g * q.gin + c) * (long)q.H * q.W;
        const float* wc = w + (transposed ? ((long)(g * q.gin + c) * q.gout + oc) : ((long)p * q.gin + c)) * taps;
#pragma unroll
        for (int i = 0; i < kh; ++i) {
            const int h = oh * q.sh - q.ph + i;
#pragma unroll
            for (int j = 0; j < kw; ++j) {
                const int x = ow * q.sw - q.pw + j, k = i * kw + j;
                const float wk = wc[transposed ? taps - 1 - k : k];
                const bool inside = (unsigned)h < (unsigned)q.H && (unsigned)x < (unsigned)q.W;
                const float v = inside ? base[(long)h * q.W + x] : 0.0f;
                // A padding position's term is a zero, and adding it changes nothing (the sum starts at +0 and never
                // becomes -0) -- unless the weight (or d) is inf or NaN, which makes the term NaN: only then is it
                // computed.  (Computed always, the zeros took the primitives' full definition in nearly every wavefront.)
                const float ws = has_off ? pam_mul(wk, off) : wk;              // (the weight as the product sees it)
                // (EXACT: the slope of a weight of 2^127 and more can be inf, and inf times the zero NaN)
                const bool finite = (f2u(ws) & 0x7fffffffu) < (EXACT ? 0x7f000000u : 0x7f800000u) && (!EXACT || (f2u(dv) & 0x7f800000u) != 0x7f800000u);
                if (inside || !finite)
                    acc = acc + (EXACT ? pam_mul_bwd(dv, wk, v, off, has_off != 0) : pam_mul(ws, v));
            }
        }
    }
    out[idx] = acc;
}

// dw[b][co][k], k = (c, i, j) of the filter's group, = sum over the output positions l of term(dy[b][co][l], x patch
// entry (k, l)), l ascending in chunks of `chunk` whose sums are added in ascending order from +0 (the order the matrix
// kernel's plan gives this sum).  EXACT false: term = (dy (*) off) (*) v; EXACT true: term = pam_bwd(w[co][k], v, dy)
// with the offset on v.
template <bool EXACT>
__global__ __launch_bounds__(256) void direct_conv_weight_kernel(const float* __restrict__ x, const float* __restrict__ dy, const float* __restrict__ w,
                                                                float* __restrict__ dw, long total, int filters, DirectGeom q, int chunk, float off,
                                                                int has_off)
{
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int taps = q.kh * q.kw, K = q.gin * taps;
    const long plane = total <= 0x7fffffffL ? (long)((int)idx / K) : idx / K;          // b * filters + co
    const int k = (int)(idx - plane * K), c = k / taps, i = (k % taps) / q.kw, j = k % q.kw;
    const int co = (int)(plane % filters), L = q.ho * q.wo;
    const long b = plane / filters;
    const float* base = x + (b * q.IC + (co / q.gout) * q.gin + c) * (long)q.H * q.W;
    const float* g = dy + plane * L;
    const float wk = EXACT ? w[(long)co * K + k] : 0.0f;
    float sum = 0.0f;
    for (int l0 = 0; l0 < L; l0 += chunk) {
        float part = 0.0f;
        const int end = min(L, l0 + chunk);
        // eight positions' loads in flight at a time (there are few lanes, each with a long chain of sums); the terms
        // are added one by one in ascending order all the same
        constexpr int kAhead = 8;
        for (int lb = l0; lb < end; lb += kAhead) {
            float v[kAhead], gv[kAhead]; bool in[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int l = min(lb + u, end - 1);
                const int h = (l / q.wo) * q.sh - q.ph + i, xx = (l % q.wo) * q.sw - q.pw + j;
                in[u] = (unsigned)h < (unsigned)q.H && (unsigned)xx < (unsigned)q.W;
                v[u] = in[u] ? base[(long)h * q.W + xx] : 0.0f; gv[u] = g[l];
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                if (lb + u >= end) break;
                const float gl = gv[u];
                // (a padding position's term is a zero unless the gradient -- or w -- is inf or NaN: see direct_conv_kernel)
                const float gs = !EXACT && has_off ? pam_mul(gl, off) : gl;     // (the gradient as the approximate product sees it)
                const bool finite = (f2u(gs) & 0x7f800000u) != 0x7f800000u && (!EXACT || (f2u(wk) & 0x7f800000u) != 0x7f800000u);
                if (in[u] || !finite)
                    part = part + (EXACT ? pam_mul_bwd(wk, v[u], gl, off, has_off != 0) : pam_mul(gs, v[u]));
            }
        }
        sum = chunk >= L ? part : sum + part;
    }
    dw[idx] = sum;
}

template <bool EXACT>
void launch_direct_conv(const float* img, const float* w, const float* d, float* out, long total, int planes, const DirectGeom& q,
                        int transposed, float off, hipStream_t st)
{
    const dim3 grid((unsigned)((total + 255) / 256));
    const int has_off = off != 1.0f ? 1 : 0, side = q.kh == q.kw ? q.kh : 0;
#define PAM_DIRECT_SIDE(S) hipLaunchKernelGGL((direct_conv_kernel<EXACT, S>), grid, dim3(256), 0, st, img, w, d, out, total, planes, q, transposed, off, has_off)
    if (side == 3) PAM_DIRECT_SIDE(3); else if (side == 5) PAM_DIRECT_SIDE(5); else if (side == 7) PAM_DIRECT_SIDE(7); else PAM_DIRECT_SIDE(0);
#undef PAM_DIRECT_SIDE
}

// Which grouped convolutions: groups of up to kDirectGroup channels and filters whose sums (either way round) are short
// enough to never be cut along k.  Depthwise only: with four channels and filters per group (32 images of 128 x 28 x 28,
// 3 x 3) the forward ran 116 us here against 125 us on the matrix kernel, but the weight gradient 295 against 117.
constexpr long kDirectGroup = 1;
bool direct_conv(const ConvShape& s)
{
    return s.g > 1 && s.cg() <= kDirectGroup && s.cog() <= kDirectGroup && s.K() < 128 && s.cog() * s.kh * s.kw < 128;
}
DirectGeom direct_geom(const ConvShape& s)
{
    return DirectGeom{(int)s.c, (int)s.h, (int)s.w, (int)s.ho, (int)s.wo, (int)s.kh, (int)s.kw, (int)s.sh, (int)s.sw, (int)s.ph, (int)s.pw,
                      (int)s.cg(), (int)s.cog()};
}

// ---------------------------------------------------------------- scratch that the library owns
// For callers that cannot allocate (code under graph capture, serving loops, harnesses that forbid hipMalloc):
// the split-k partial tiles of pam_hip_pam_matmul_fwd_noalloc go to this array instead of a workspace argument.
// Every GPU the library runs on holds its own copy, at its own address, until the process ends.
constexpr size_t kScratchBytes = (size_t)PAM_HIP_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// The array's address on the current device.  In host code `scratch` is only a stand-in for the symbol, never an
// address to hand to a kernel; the address is looked up once per device, with that device current.
int scratch_address(const char* what, void** ptr)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return pamhost::fail(PAM_HIP_ERR_LAUNCH, "%s: hipGetDevice: %s", what, hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "%s: device %d beyond the %d this entry point keeps scratch for", what, dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return pamhost::fail(PAM_HIP_ERR_LAUNCH, "%s: hipGetSymbolAddress: %s", what, hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *ptr = g_scratch_ptr[dev];
    return PAM_HIP_OK;
}

}  // namespace

extern "C" {

size_t pam_hip_gemm_workspace_bytes(long batch, long m, long n, long k)
{
    if (batch <= 0 || m <= 0 || n <= 0 || k <= 0) return 0;
    return plan_space(make_plan(batch, m, n, k, true)).total;
}

void pam_hip_set_tuning(int bk, int pieces) { g_force_bk = bk; g_force_pieces = pieces; }

int pam_hip_gemm_priority_steps(long batch, long m, long n, long k, int exact)
{
    if (batch <= 0 || m <= 0 || n <= 0 || k < 0) return 0;
    return priority_steps(launch_plan(make_plan(batch, m, n, k > 0 ? k : 1, true), exact == 0, false, true, batch, m, n, k), m, n, exact != 0) ? 1 : 0;
}

int pam_hip_gemm_schedule(long batch, long m, long n, long k, int kind, int* k_tile, int* tile_rows, int* tile_columns, long* work_groups)
{
    if (batch <= 0 || m <= 0 || n <= 0 || k <= 0 || kind < 0 || kind > 2 || !k_tile || !tile_rows || !tile_columns || !work_groups)
        return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "gemm_schedule: bad shape, kind or null pointer");
    const Plan p = launch_plan(make_plan(batch, m, n, k, true), kind == 0, kind == 2, true, batch, m, n, k);
    *k_tile = p.bk; *work_groups = p.units;
    *tile_rows = p.free.r > 0 ? 4 * p.free.r : 64; *tile_columns = p.free.r > 0 ? 4 * p.free.c : 64;
    return PAM_HIP_OK;
}

int pam_hip_gemm_plan(long batch, long m, long n, long k, int* k_chunk)
{
    if (batch <= 0 || m <= 0 || n <= 0 || k < 0) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "gemm_plan: bad shape");
    Plan p = make_plan(batch, m, n, k > 0 ? k : 1, true);
    if (k_chunk) *k_chunk = p.piece_kt * p.bk;
    return PAM_HIP_OK;
}

int pam_hip_pam_matmul_fwd(const float* a, long a_sr, long a_sc, const float* b, long b_sr, long b_sc,
                           float* y, long y_sr, long y_sc, long m, long n, long k, float offset,
                           void* workspace, size_t workspace_bytes, void* stream)
{
    return gemm("pam_matmul_fwd", MODE_PAM, 1, m, n, k, a, 0, a_sr, a_sc, b, 0, b_sr, b_sc, nullptr, 0, 0, 0,
                y, 0, y_sr, y_sc, offset, workspace, workspace_bytes, stream);
}

int pam_hip_pam_matmul_fwd_noalloc(const float* a, long a_sr, long a_sc, const float* b, long b_sr, long b_sc,
                                   float* y, long y_sr, long y_sc, long m, long n, long k, float offset, void* stream)
{
    const size_t need = pam_hip_gemm_workspace_bytes(1, m, n, k);
    if (need > kScratchBytes)
        return pamhost::fail(PAM_HIP_ERR_WORKSPACE, "pam_matmul_fwd_noalloc: this shape needs %zu bytes of scratch, the library holds %zu; "
                             "use pam_hip_pam_matmul_fwd with a workspace", need, kScratchBytes);
    void* ws = nullptr;
    if (need > 0) {
        const int rc = scratch_address("pam_matmul_fwd_noalloc", &ws);
        if (rc != PAM_HIP_OK) return rc;
    }
    return gemm("pam_matmul_fwd_noalloc", MODE_PAM, 1, m, n, k, a, 0, a_sr, a_sc, b, 0, b_sr, b_sc, nullptr, 0, 0, 0,
                y, 0, y_sr, y_sc, offset, ws, need, stream);
}

int pam_hip_pam_linear_fwd(const float* a, long a_sr, long a_sc, const float* b, long b_sr, long b_sc, const float* bias,
                           float* y, long y_sr, long y_sc, long m, long n, long k, float offset,
                           void* workspace, size_t workspace_bytes, void* stream)
{
    return gemm("pam_linear_fwd", MODE_PAM, 1, m, n, k, a, 0, a_sr, a_sc, b, 0, b_sr, b_sc, nullptr, 0, 0, 0,
                y, 0, y_sr, y_sc, offset, workspace, workspace_bytes, stream, nullptr, bias);
}

int pam_hip_pam_bmm_fwd(PAM_HIP_MAT(a), PAM_HIP_MAT(b), PAM_HIP_OUT(y), long batch, long m, long n, long k,
                        float offset, void* workspace, size_t workspace_bytes, void* stream)
{
    return gemm("pam_bmm_fwd", MODE_PAM, batch, m, n, k, a, a_sb, a_sr, a_sc, b, b_sb, b_sr, b_sc, nullptr, 0, 0, 0,
                y, y_sb, y_sr, y_sc, offset, workspace, workspace_bytes, stream);
}

int pam_hip_standard_matmul(const float* a, long a_sr, long a_sc, const float* b, long b_sr, long b_sc,
                            float* y, long y_sr, long y_sc, long m, long n, long k, float ignored,
                            void* workspace, size_t workspace_bytes, void* stream)
{
    (void)ignored;
    return gemm("standard_matmul", MODE_STD, 1, m, n, k, a, 0, a_sr, a_sc, b, 0, b_sr, b_sc, nullptr, 0, 0, 0,
                y, 0, y_sr, y_sc, 1.0f, workspace, workspace_bytes, stream);
}

int pam_hip_standard_bmm(PAM_HIP_MAT(a), PAM_HIP_MAT(b), PAM_HIP_OUT(y), long batch, long m, long n, long k,
                         float ignored, void* workspace, size_t workspace_bytes, void* stream)
{
    (void)ignored;
    return gemm("standard_bmm", MODE_STD, batch, m, n, k, a, a_sb, a_sr, a_sc, b, b_sb, b_sr, b_sc, nullptr, 0, 0, 0,
                y, y_sb, y_sr, y_sc, 1.0f, workspace, workspace_bytes, stream);
}

int pam_hip_pam_matmul_bwd(const float* l, long l_sr, long l_sc, const float* r, long r_sr, long r_sc,
                           const float* mo, long mo_sr, long mo_sc, float* dm, long dm_sr, long dm_sc,
                           long m, long n, long k, int delta_l, float offset,
                           void* workspace, size_t workspace_bytes, void* stream)
{
    return gemm("pam_matmul_bwd", delta_l ? MODE_BWD_DL : MODE_BWD_DR, 1, m, n, k, l, 0, l_sr, l_sc, r, 0, r_sr, r_sc,
                mo, 0, mo_sr, mo_sc, dm, 0, dm_sr, dm_sc, offset, workspace, workspace_bytes, stream);
}

int pam_hip_pam_bmm_bwd(PAM_HIP_MAT(l), PAM_HIP_MAT(r), PAM_HIP_MAT(mo), PAM_HIP_OUT(dm),
                        long batch, long m, long n, long k, int delta_l, float offset,
                        void* workspace, size_t workspace_bytes, void* stream)
{
    return gemm("pam_bmm_bwd", delta_l ? MODE_BWD_DL : MODE_BWD_DR, batch, m, n, k, l, l_sb, l_sr, l_sc, r, r_sb, r_sr, r_sc,
                mo, mo_sb, mo_sr, mo_sc, dm, dm_sb, dm_sr, dm_sc, offset, workspace, workspace_bytes, stream);
}

size_t pam_hip_conv2d_workspace_bytes(long batch, long c, long h, long w, long co, long kh, long kw,
                                      long stride_h, long stride_w, long pad_h, long pad_w, long groups, int which, float offset)
{
    ConvShape s{batch, c, h, w, co, kh, kw, stride_h, stride_w, pad_h, pad_w, 0, 0, groups};
    if (conv_shape("conv2d_workspace_bytes", s) != PAM_HIP_OK || batch == 0) return 0;
    if (which == 2) {
        ConvShape t;
        if (input_gradient_shape("conv2d_workspace_bytes", s, t) != PAM_HIP_OK) return 0;
        return input_gradient_space(t).total;
    }
    // (1: the larger of the two weight gradients' needs, whichever the caller then asks for)
    if (which == 1) return std::max(conv_space(s, 1, offset != 1.0f).total, conv_space(s, 2, false).total);
    return conv_space(s, 0, offset != 1.0f).total;
}

int pam_hip_conv2d_bwd_input(const float* dy, const float* w, const float* x, float* dx, long batch, long c, long h, long wd,
                             long co, long kh, long kw, long stride_h, long stride_w, long pad_h, long pad_w, long groups,
                             int exact, float offset, void* workspace, size_t workspace_bytes, void* stream)
{
    ConvShape s{batch, c, h, wd, co, kh, kw, stride_h, stride_w, pad_h, pad_w, 0, 0, groups};
    int rc = conv_shape("conv2d_bwd_input", s);
    if (rc != PAM_HIP_OK) return rc;
    ConvShape t;
    rc = input_gradient_shape("conv2d_bwd_input", s, t);
    if (rc != PAM_HIP_OK) return rc;
    if (batch == 0) return PAM_HIP_OK;
    if (!dy || !w || !dx || (exact && !x)) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "conv2d_bwd_input: null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (direct_conv(s)) {                             // the convolution of dy with the flipped weights, directly
        const long total = batch * c * h * wd;
        if (total >= (1L << 31) * 256) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "conv2d_bwd_input: too many outputs");
        const DirectGeom q = direct_geom(t);          // (t: the image is dy, a group's sums run over its filters)
        if (exact) launch_direct_conv<true>(dy, w, x, dx, total, (int)c, q, 1, offset, st);
        else launch_direct_conv<false>(dy, w, nullptr, dx, total, (int)c, q, 1, offset, st);
        return pamhost::check_launch("conv2d_bwd_input");
    }
    ConvSpace sp = input_gradient_space(t);
    ConvGeom cv;
    rc = conv_prepare("conv2d_bwd_input", t, sp, workspace, workspace_bytes, st, cv, false);
    if (rc != PAM_HIP_OK) return rc;
    float* wf = (float*)((char*)workspace + sp.tables);
    const bool one_launch = replicated(t);
    const long copies = one_launch ? batch : 1;
    const long n = c * s.cog() * kh * kw * copies;
    // approximate: the offset goes into the flipped weights; exact: the product kernel applies it to its slope operand
    hipLaunchKernelGGL(flip_weights_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, w, wf, (int)c, (int)s.cog(), (int)s.cg(),
                       (int)kh, (int)kw, offset, (!exact && offset != 1.0f) ? 1 : 0, (int)copies);
    const long K = t.K(), L = t.L();                  // K = (co / groups) kh kw, L = h w
    void* rest = (char*)workspace + sp.tables + sp.scaled; size_t rest_bytes = workspace_bytes - sp.tables - sp.scaled;
    const long hw_out = s.ho * s.wo;
    if (one_launch) {                                 // unit z = image * groups + group (see kReplicateBytes)
        if (exact)
            return gemm("conv2d_bwd_input", MODE_BWD_DR, batch * groups, s.cg(), L, K, wf, s.cg() * K, K, 1, dy, s.cog() * hw_out, 0, 0,
                        x, s.cg() * L, L, 1, dx, s.cg() * L, L, 1, offset, rest, rest_bytes, stream, &cv);
        return gemm("conv2d_bwd_input", MODE_PAM, batch * groups, s.cg(), L, K, wf, s.cg() * K, K, 1, dy, s.cog() * hw_out, 0, 0,
                    nullptr, 0, 0, 0, dx, s.cg() * L, L, 1, 1.0f, rest, rest_bytes, stream, &cv);
    }
    for (long gi = 0; gi < groups; ++gi) {            // one product per group: its filters' gradient slices in, its channels out
        const float* wg = wf + gi * s.cg() * K;
        const float* dyg = dy + gi * s.cog() * hw_out;
        float* dxg = dx + gi * s.cg() * L;
        if (exact)    // dX[c, l] = sum_k pam_bwd(x[c, l], wf[c, k], dY patch[k, l]): x is the same for every term of an output
            rc = gemm("conv2d_bwd_input", MODE_BWD_DR, batch, s.cg(), L, K, wg, 0, K, 1, dyg, co * hw_out, 0, 0, x + gi * s.cg() * L, c * L, L, 1,
                      dxg, c * L, L, 1, offset, rest, rest_bytes, stream, &cv);
        else
            rc = gemm("conv2d_bwd_input", MODE_PAM, batch, s.cg(), L, K, wg, 0, K, 1, dyg, co * hw_out, 0, 0, nullptr, 0, 0, 0,
                      dxg, c * L, L, 1, 1.0f, rest, rest_bytes, stream, &cv);
        if (rc != PAM_HIP_OK) return rc;
    }
    return PAM_HIP_OK;
}

int pam_hip_conv2d_fwd(const float* x, const float* w, float* y, long batch, long c, long h, long wd, long co, long kh, long kw,
                       long stride_h, long stride_w, long pad_h, long pad_w, long groups, float offset,
                       void* workspace, size_t workspace_bytes, void* stream)
{
    ConvShape s{batch, c, h, wd, co, kh, kw, stride_h, stride_w, pad_h, pad_w, 0, 0, groups};
    int rc = conv_shape("conv2d_fwd", s);
    if (rc != PAM_HIP_OK) return rc;
    if (batch == 0) return PAM_HIP_OK;
    if (!x || !w || !y) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "conv2d_fwd: null pointer");
    hipStream_t st = (hipStream_t)stream;
    const bool has_off = offset != 1.0f;
    if (direct_conv(s)) {
        const long total = batch * co * s.L();
        if (total >= (1L << 31) * 256) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "conv2d_fwd: too many outputs");
        launch_direct_conv<false>(x, w, nullptr, y, total, (int)co, direct_geom(s), 0, offset, st);
        return pamhost::check_launch("conv2d_fwd");
    }
    ConvSpace sp = conv_space(s, 0, has_off);
    ConvGeom cv;
    rc = conv_prepare("conv2d_fwd", s, sp, workspace, workspace_bytes, st, cv, false);
    if (rc != PAM_HIP_OK) return rc;
    // the reference folds the offset into the weights (the right operand of its product); here the
    // weights are the left operand, so they are scaled once up front
    const float* wl = w;
    const bool one_launch = replicated(s);
    if (has_off || one_launch) {
        float* scaled = (float*)((char*)workspace + sp.tables);
        launch_scale(w, scaled, (size_t)co * s.K(), one_launch ? (size_t)batch : 1, offset, has_off, st);
        wl = scaled;
    }
    const long K = s.K(), L = s.L();
    if (one_launch)                                   // unit z = image * groups + group (see kReplicateBytes)
        return gemm("conv2d_fwd", MODE_PAM, batch * groups, s.cog(), L, K, wl, s.cog() * K, K, 1, x, s.cg() * h * wd, 0, 0,
                    nullptr, 0, 0, 0, y, s.cog() * L, L, 1, 1.0f,
                    (char*)workspace + sp.tables + sp.scaled, workspace_bytes - sp.tables - sp.scaled, stream, &cv);
    // per image and group: Y[co, l] = sum_k W[co, k] (*) patches[k, l] over the group's channels
    for (long gi = 0; gi < groups; ++gi) {
        rc = gemm("conv2d_fwd", MODE_PAM, batch, s.cog(), L, K, wl + gi * s.cog() * K, 0, K, 1, x + gi * s.cg() * h * wd, c * h * wd, 0, 0,
                  nullptr, 0, 0, 0, y + gi * s.cog() * L, co * L, L, 1, 1.0f,
                  (char*)workspace + sp.tables + sp.scaled, workspace_bytes - sp.tables - sp.scaled, stream, &cv);
        if (rc != PAM_HIP_OK) return rc;
    }
    return PAM_HIP_OK;
}

int pam_hip_conv2d_bwd_weight(const float* x, const float* dy, const float* w, float* dw, long batch, long c, long h, long wd,
                              long co, long kh, long kw, long stride_h, long stride_w, long pad_h, long pad_w, long groups,
                              int exact, float offset, void* workspace, size_t workspace_bytes, void* stream)
{
    ConvShape s{batch, c, h, wd, co, kh, kw, stride_h, stride_w, pad_h, pad_w, 0, 0, groups};
    int rc = conv_shape("conv2d_bwd_weight", s);
    if (rc != PAM_HIP_OK) return rc;
    if (batch == 0) return PAM_HIP_OK;
    if (!x || !dy || !dw || (exact && !w)) return pamhost::fail(PAM_HIP_ERR_ARGUMENT, "conv2d_bwd_weight: null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (direct_conv(s)) {
        // the sum over the output positions in the chunks the matrix kernel would cut it into (given its workspace)
        const Plan p = make_plan(batch * groups, s.cog(), s.K(), s.L(), true);
        const int chunk = p.pieces > 1 ? p.piece_kt * p.bk : (int)std::min<long>(s.L(), 1L << 30);
        const long total = batch * co * s.K();
        const dim3 grid((unsigned)((total + 255) / 256));
        if (exact) hipLaunchKernelGGL(direct_conv_weight_kernel<true>, grid, dim3(256), 0, st, x, dy, w, dw, total, (int)co, direct_geom(s), chunk, offset, offset != 1.0f ? 1 : 0);
        else hipLaunchKernelGGL(direct_conv_weight_kernel<false>, grid, dim3(256), 0, st, x, dy, (const float*)nullptr, dw, total, (int)co, direct_geom(s), chunk, offset, offset != 1.0f ? 1 : 0);
        return pamhost::check_launch("conv2d_bwd_weight");
    }
    const bool scale = offset != 1.0f && !exact;
    ConvSpace sp = conv_space(s, exact ? 2 : 1, scale);
    ConvGeom cv;
    rc = conv_prepare("conv2d_bwd_weight", s, sp, workspace, workspace_bytes, st, cv, true);
    if (rc != PAM_HIP_OK) return rc;
    const long K = s.K(), L = s.L();
    void* rest = (char*)workspace + sp.tables + sp.scaled; size_t rest_bytes = workspace_bytes - sp.tables - sp.scaled;
    // approximate: dW[co, k] = sum_l patches[k, l] (*) (dY[co, l] (*) offset), the gradient scaled once up front
    const float* dl = dy;
    if (scale) {
        float* scaled = (float*)((char*)workspace + sp.tables);
        launch_scale(dy, scaled, (size_t)batch * co * L, 1, offset, true, st);
        dl = scaled;
    }
    // grouped: unit z = image * groups + group (see kReplicateBytes); only the exact gradient reads the weights
    if (groups > 1 && !exact)
        return gemm("conv2d_bwd_weight", MODE_PAM, batch * groups, s.cog(), K, L, dl, s.cog() * L, L, 1, x, s.cg() * h * wd, 0, 0,
                    nullptr, 0, 0, 0, dw, s.cog() * K, K, 1, 1.0f, rest, rest_bytes, stream, &cv);
    if (groups > 1 && replicated(s)) {
        float* copies = (float*)((char*)workspace + sp.tables);
        launch_scale(w, copies, (size_t)co * K, (size_t)batch, 1.0f, false, st);
        return gemm("conv2d_bwd_weight", MODE_BWD_DL, batch * groups, s.cog(), K, L, dy, s.cog() * L, L, 1, x, s.cg() * h * wd, 0, 0,
                    copies, s.cog() * K, K, 1, dw, s.cog() * K, K, 1, offset, rest, rest_bytes, stream, &cv);
    }
    for (long gi = 0; gi < groups; ++gi) {
        const float* xg = x + gi * s.cg() * h * wd;
        float* dwg = dw + gi * s.cog() * K;
        if (exact)    // dW[co, k] = sum_l pam_bwd(W[co, k], patches[k, l], dY[co, l]); the offset goes with the patches
            rc = gemm("conv2d_bwd_weight", MODE_BWD_DL, batch, s.cog(), K, L, dy + gi * s.cog() * L, co * L, L, 1, xg, c * h * wd, 0, 0,
                      w + gi * s.cog() * K, 0, K, 1, dwg, co * K, K, 1, offset, rest, rest_bytes, stream, &cv);
        else
            rc = gemm("conv2d_bwd_weight", MODE_PAM, batch, s.cog(), K, L, dl + gi * s.cog() * L, co * L, L, 1, xg, c * h * wd, 0, 0,
                      nullptr, 0, 0, 0, dwg, co * K, K, 1, 1.0f, rest, rest_bytes, stream, &cv);
        if (rc != PAM_HIP_OK) return rc;
    }
    return PAM_HIP_OK;
}

}  // extern "C"
