// Tiled MFMA GEMM family for gfx950: which problems the kernels take, and the choice of the instantiation.
// The kernel template is gemm_tile_kernel.h; gemm_tile_<kind>_<layout>.hip instantiate it.
#include <algorithm>
#include <cmath>

#include "common.h"
#include "gemm_common.h"
#include "gemm_mid.h"
#include "gemm_stream.h"
#include "gemm_tail.h"
#include "gemm_tile_shape.h"

namespace cch {

template <int KIND, int EPI, int FMT, int TB> int launch_tile_t(const GemmProblem &p, hipStream_t stream);
template <int KIND, int EPI, int FMT, int TB> int launch_stream_t(const GemmProblem &p, int waves, hipStream_t stream);
template <int KIND, int EPI, int FMT, int TB> int launch_mid_t(const GemmProblem &p, int rows, int cols, hipStream_t stream);
#define CCH_TILE_FAMILY(KIND, EPI, FMT) \
    extern template int launch_tile_t<KIND, EPI, FMT, 0>(const GemmProblem &, hipStream_t); \
    extern template int launch_tile_t<KIND, EPI, FMT, 1>(const GemmProblem &, hipStream_t); \
    extern template int launch_stream_t<KIND, EPI, FMT, 0>(const GemmProblem &, int, hipStream_t); \
    extern template int launch_stream_t<KIND, EPI, FMT, 1>(const GemmProblem &, int, hipStream_t); \
    extern template int launch_mid_t<KIND, EPI, FMT, 0>(const GemmProblem &, int, int, hipStream_t); \
    extern template int launch_mid_t<KIND, EPI, FMT, 1>(const GemmProblem &, int, int, hipStream_t);
CCH_TILE_FAMILY(KIND_I8, EPI_DEQUANT, 0)
CCH_TILE_FAMILY(KIND_I8, EPI_DEQUANT_SWIGLU, 0)
CCH_TILE_FAMILY(KIND_F8, EPI_PLAIN, CCH_FMT_E4M3)
CCH_TILE_FAMILY(KIND_F8, EPI_PLAIN, CCH_FMT_E5M2)
CCH_TILE_FAMILY(KIND_F8, EPI_SWIGLU, CCH_FMT_E4M3)
CCH_TILE_FAMILY(KIND_F8, EPI_SWIGLU, CCH_FMT_E5M2)
CCH_TILE_FAMILY(KIND_F4, EPI_PLAIN, CCH_FMT_E2M1)
CCH_TILE_FAMILY(KIND_F4, EPI_SWIGLU, CCH_FMT_E2M1)
#undef CCH_TILE_FAMILY

#ifdef CCH_PROF
// Measurement build: counters of the last tiled launch (see gemm_tile_kernel.h).
int (*g_prof_copy)(uint64_t *, int) = nullptr;
extern "C" int cch_prof_read(uint64_t *host) { return g_prof_copy ? g_prof_copy(host, 0) : -1; }
extern "C" int cch_prof_read_tiles(uint64_t *host) { return g_prof_copy ? g_prof_copy(host, 1) : -1; }
extern "C" int cch_prof_read_entry(uint64_t *host) { return g_prof_copy ? g_prof_copy(host, 2) : -1; }
#endif

// nullptr when the tiled kernels take this problem; otherwise the precondition that failed (the
// caller then uses the generic path or reports it).
const char *gemm_tile_unsupported(const GemmProblem &p, int kind, int epi)
{
    const int epb = kind == KIND_F4 ? 2 : 1;
    const int64_t lda = p.K / epb;
    // rows are fetched in 16-byte pieces
    if (p.K < 1 || p.K % (16 * epb) != 0) return "K must be a multiple of 16 bytes per row";
    if (p.n_out % 8 != 0 || !aligned(p.out, 16)) return "output rows must take 16-byte stores (n_out % 8 == 0, out 16-byte aligned)";
    if (p.mx_out && ((epi != EPI_DEQUANT_SWIGLU && epi != EPI_SWIGLU) || p.n_out % 32 != 0 || p.out_fp16)) return "MX-quantised output needs whole 32-column blocks";
    if ((int64_t)BM * p.n_out * 2 >= ((int64_t)1 << 31)) return "output row tile beyond 2 GiB";
    // mapped output rows are addressed from the start of `out` with 32-bit offsets
    if (p.out_row_map && (epi != EPI_PLAIN || p.out_rows * p.n_out * 2 >= ((int64_t)1 << 31) || !aligned(p.out_row_map, 4)))
        return "mapped output beyond 2 GiB or misaligned row map";
    if (p.num_groups > MAX_GROUPS) return "more than 256 groups";
    if ((int64_t)p.N * lda >= ((int64_t)1 << 31)) return "one right-hand operand beyond 2 GiB (32-bit source offsets)";
    if ((int64_t)BM * std::max<int64_t>(lda, p.a_pitch) >= ((int64_t)1 << 31)) return "a row tile of the left-hand operand beyond 2 GiB";
    // (the 16-byte requests need dword alignment only: packed rows of K = 256 are 264 bytes long)
    if (p.a_pitch && (p.a_pitch % 4 != 0 || p.a_pitch < lda)) return "rows of the left-hand operand must start on 4-byte boundaries";
    if (p.sa_pitch && (p.sa_pitch % 2 != 0 || p.sa_pitch < p.sld)) return "scale rows of the left-hand operand must start on even addresses";
    if (!aligned(p.a, 16) || !aligned(p.b, 16) || p.b_stride % 16 != 0) return "operands must be 16-byte aligned";
    if (kind != KIND_I8 && (!aligned(p.sa, 4) || !aligned(p.sb, 4) || p.sb_stride % 2 != 0)) return "scale arrays must be 4-byte aligned";
    if (kind != KIND_I8 && ((int64_t)p.num_groups * p.N * p.sld >= ((int64_t)1 << 31) || (int64_t)p.T * std::max<int64_t>(p.sld, p.sa_pitch) >= ((int64_t)1 << 31)))
        return "scale arrays beyond 2 GiB";
    if (kind != KIND_I8 && p.sb_stride != (int64_t)p.N * p.sld) return "scale arrays of the right-hand operands must be back to back";
    if ((epi == EPI_DEQUANT || epi == EPI_DEQUANT_SWIGLU) && (!aligned(p.per_tok, 4) || !aligned(p.per_ch, 4))) return "dequantisation scales must be 4-byte aligned";
    if (!p.trans_b) {
        // [K, N] operands: rows of B are fetched in 16-byte pieces that start on 4-byte boundaries
        if ((p.N / epb) % 4 != 0) return "[K,N] operands need rows of a multiple of 4 bytes";
        if ((epi == EPI_DEQUANT_SWIGLU || epi == EPI_SWIGLU) && (p.n_out / epb) % 4 != 0) return "[K,N] SwiGLU operands need n/2 to be a multiple of 4";
    }
    return nullptr;
}

// ---- which of the kernels takes a problem
//
// The 256 x 256 tiles have the fewest bytes through L2 and LDS per product, and one persistent workgroup per CU; the smaller
// tiles of the others fill more CUs, in shorter steps.  What decides is how many tiles there are to a CU and how long K is, so
// each kernel has an estimate of its time,
//     us = start + max(steps * max(step_alone, step_full * fill) + finish * fill, weights * per_mb),
//     steps: 128-byte steps of K one wave walks, fill: tiles / CUs, weights: MB of right-hand operands,
// and the smallest one wins (the 256 x 256 kernel unless another is estimated 8 % faster).  With one workgroup to a CU a last,
// partly empty round costs at least half a full one: fill counts as floor(fill) + 0.5 + 0.5 * the rest.  The constants are fits of this form by
// the choices they lead to, not by the times, which are off by 10 to 20 % each: the table's first to 1200 problems (dense and grouped, all kinds
// and layouts), GROUPED_TILE to 6100 groupings of 3800 others.
// The sizes of groups are not known here: fill counts average groups, whose last row tile is half full.  With [N, K] weights, which come to
// the 256 x 256 kernel at a rate that depends on the CUs at work, that was not enough for its time, which goes up in whole rounds:
// 128 rows of each of 16 experts are one row tile each if the groups are alike and 1.1 if they are skewed, and with 16 column tiles that is one round of
// the chip or the start of another.  There its estimate is the mean of one for groups alike (spread as far as a random routing spreads them)
// and one for skewed groups (any size up to twice the average), each over the row tiles more or less that so many groups come to.
// On 1300 problems that nothing was fitted to (times of every kernel in profiles/gemm_kernel_times.csv, 1900 groupings) the choices are within
// 2.6 % of the best kernel in the geometric mean (dense 1.6, grouped 2.7), take 0.72 of the 256 x 256 kernel's time (dense 0.46, grouped 0.76) and
// are more than 10 % slower than that kernel on 18 groupings; with one estimate for average groups and a rate of weights that changed where a second launch
// is tried on 21, and on 170 of 2500 groupings with [N, K] weights and many near whole rounds, now 79.  Of 2374 products of perf/cases.py's ranges 5 got
// slower by more than 3 % and 3 faster.  (The same form for [K, N] weights too, or all constants fitted anew, per operand kind, gained more near whole rounds
// and lost elsewhere: 18 and 51 of the 2374 slower by more than 3 %.)
struct PathModel {
    int tm, tn, waves_k;    // rows and columns of B per tile, waves that share a tile's K
    bool rounds;            // a CU runs one workgroup at a time, and tiles long enough for that to count
    double start, step_alone, step_full, finish;
    double per_mb[3];       // B as [N, K], as [K, N], and as [K, N] with gate and up columns apart (narrower pieces of a row)
};
static const PathModel PATH_MODEL[NUM_KERNELS] = {
    {256, 256, 1, true, 9.7, 1.27, 1.66, 3.9, {0.30, 0.20, 0.21}},
    {64, 128, 1, false, 4.5, 0.37, 0.50, 1.55, {0.18, 0.22, 0.22}},
    {128, 128, 1, false, 5.75, 0.48, 0.65, 1.55, {0.19, 0.22, 0.27}},
    {128, 256, 1, true, 5.6, 0.69, 1.07, 4.9, {0.20, 0.22, 0.205}},
    {STREAM_TM, STREAM_TN, 4, false, 3.35, 0.95, 1.09, 1.05, {0.245, 0.29, 0.30}},
    {STREAM_TM, STREAM_TN, 8, false, 3.7, 1.24, 1.92, 2.0, {0.21, 0.255, 0.46}},
};
// The 256 x 256 kernel on grouped problems with [N, K] weights: every round started costs a whole `finish`.
static const PathModel GROUPED_TILE = {256, 256, 1, true, 9.93, 1.22, 1.36, 4.34, {0.233, 0.0, 0.0}};

// Average of the row tiles of a group whose size lies anywhere in [lo, hi] rows, tiles of tm rows; a group has at least one.
static double row_tiles_of(double lo, double hi, int tm)
{
    auto sum = [](double x) {   // integral of ceil from 0
        const double n = std::floor(x);
        return n * (n + 1) / 2 + (x - n) * (n + 1);
    };
    return std::max(1.0, (sum(hi / tm) - sum(lo / tm)) * tm / (hi - lo));
}

// us of the 256 x 256 kernel on a grouped problem with [N, K] weights.
static double grouped_tile_us(const GemmProblem &p, double steps, double weights, int tn_out, int cus)
{
    const PathModel &m = GROUPED_TILE;
    const double groups = std::min<int64_t>(p.num_groups, p.T), average = p.T / groups, spread = 1.73 * std::sqrt(average);
    const double per_row_tile = (double)((p.n_out + tn_out - 1) / tn_out) / cus, more_or_less = 0.5 * std::sqrt(groups);
    const double row_tiles[2] = {groups * row_tiles_of(std::max(0.0, average - spread), average + spread, m.tm),
                                 groups * row_tiles_of(0.0, 2 * average, m.tm)};
    double us = 0.0;
    for (double tiles : row_tiles)
        for (int d = -7; d <= 7; d += 2) {
            const double fill = std::max(tiles + d / 8.0 * more_or_less, groups) * per_row_tile, whole = std::floor(fill), rest = fill - whole;
            const double rounds = fill > 1.0 && rest > 0.0 ? whole + 0.5 + 0.5 * rest : fill, started = fill > 1.0 ? std::ceil(fill) : fill;
            us += m.start + std::max(steps * std::max(m.step_alone, m.step_full * rounds) + m.finish * started, weights * m.per_mb[0]);
        }
    return us / 16;
}

// Whether a grouped problem on 256 x 256 tiles leaves the short row tiles of its last round to a second launch (gemm_tail.h; the device
// decides which, if any).  Worth it behind one round of long tiles, which the second, mostly empty round would nearly double: MXFP8,
// 16 groups of 3072 rows in all, K 7168, N 4096 (1.12 to 1.19 rounds) 156-177 -> 150-159 us, 8 of 4096, K 4096 (1.25) 87-91 -> 80-83.  Behind
// two rounds, or with 2048 of K, the second launch's start and the weights it reads again cost what it saves (84 against 79-87 us; int8 at
// 2.4 rounds 258 against 254).  SwiGLU weights stored [K, N] reach its narrow tiles in pieces of 64 bytes: of the measured problems in this
// window that have a second launch, 10 of those were 7 % slower with it on average, 20 with plain [K, N] weights 4 % faster, 23 with [N, K]
// ones 3 % and 15 with [N, K] SwiGLU ones 11 %.  Where the device finds nothing to leave out, the empty second launch costs 3 us.
static bool may_have_tail(const GemmProblem &p, bool swiglu, double steps, double fill)
{
    return p.group_sizes != nullptr && p.num_groups > 1 && fill > 1.0 && fill <= 1.4 && steps >= 32 &&
           (p.trans_b || (!swiglu && p.N < 1 << 21));
}

// Average number of tiles to a CU: a group's last row tile is half full on average; groups of a few rows have one tile each.
static double fill_of(const GemmProblem &p, int tm, int tn_out, int cus)
{
    const double groups = std::min<int64_t>(p.num_groups, p.T);   // that can have rows
    const double row_tiles = p.group_sizes ? std::max<double>(groups, (double)p.T / tm + 0.5 * groups) : (double)((p.T + tm - 1) / tm);
    return row_tiles * ((p.n_out + tn_out - 1) / tn_out) / cus;
}

// Scale rows of A or B that can start 2 bytes past a dword: the mid-size kernels' UA form.
static bool scales_off_dwords(const GemmProblem &p, int kind) { return kind != KIND_I8 && ((p.sld & 3) != 0 || (p.sa_pitch & 3) != 0); }

// nullptr where kernel `path` can take a problem that gemm_tile_unsupported() has let pass.
static const char *path_refuses(const GemmProblem &p, int kind, int path)
{
    if (path == PATH_TILE) return nullptr;
    // the smaller kernels add up to 512 K-rows of a [K, N] operand to offsets below 2^31
    if (!p.trans_b && p.N / (kind == KIND_F4 ? 2 : 1) >= 1 << 21) return "rows of a [K,N] operand of 2 MiB or more";
    if (path == PATH_TILE_TAIL && p.group_sizes == nullptr) return "only grouped problems have a second launch";
    if (path == PATH_MID3 && kind == KIND_F4 && scales_off_dwords(p, kind)) return "no LDS left for MXFP4 scale rows off 4-byte boundaries";
    return nullptr;
}

static GemmPath choose_path(const GemmProblem &p, int kind, int epi, int cus)
{
    const int epb = kind == KIND_F4 ? 2 : 1;
    const bool swiglu = epi == EPI_DEQUANT_SWIGLU || epi == EPI_SWIGLU;
    const double steps = (p.K / epb + BKB - 1) / BKB;
    const double groups = std::min<int64_t>(p.num_groups, p.T);   // that can have rows
    const double weights = groups * (double)p.N * (p.K / epb) * 1e-6;
    const int layout = p.trans_b ? 0 : swiglu ? 2 : 1;
    const bool tail = may_have_tail(p, swiglu, steps, fill_of(p, 256, swiglu ? 128 : 256, cus));
    GemmPath best = tail ? PATH_TILE_TAIL : PATH_TILE;
    if (path_refuses(p, kind, PATH_STREAM4)) return PATH_TILE;
    double best_us = 0.0;
    for (int i = 0; i < NUM_KERNELS; i++) {
        const PathModel &m = PATH_MODEL[i];
        const double fill = fill_of(p, m.tm, swiglu ? m.tn / 2 : m.tn, cus), whole = std::floor(fill);
        double rounds = m.rounds && fill > 1.0 && fill > whole ? whole + 0.5 + 0.5 * (fill - whole) : fill;
        // (groups: fill is an average, and a tile too many costs half a round: what that comes to over all fractions)
        if (i == PATH_MID3 && p.group_sizes && fill > 1.0) rounds = fill + 0.25;
        double us = m.start + std::max(steps / m.waves_k * std::max(m.step_alone, m.step_full * rounds) + m.finish * fill, weights * m.per_mb[layout]);
        if (i == PATH_TILE && p.group_sizes && p.trans_b) us = grouped_tile_us(p, steps, weights, swiglu ? 128 : 256, cus);
        // (with [K, N] weights the second launch is priced by itself)
        else if (i == PATH_TILE && tail)
            us = std::min(us, m.start + std::max(steps * m.step_full + m.finish * fill, weights * m.per_mb[layout]) + 5.0 + 0.45 * steps);
        if (i == PATH_TILE) {
            best_us = 0.92 * us;
        } else if (us < best_us) {
            best = (GemmPath)i;
            best_us = us;
        }
    }
    return path_refuses(p, kind, best) ? PATH_MID2 : best;   // (128 x 256 tiles: the other ones with 128 rows)
}

// Whether a problem runs on 192 x 192 tiles (gemm_mid_kernel.h; MX kinds, [N, K] weights, no activation), whatever choose_path says: where 128 x 128
// tiles, two to a CU, make more than one round and 192 x 192 ones at most one.  Measured (us, best other kernel -> this): E4M3 3000 x 1984 x 3000
// 32.9 -> 28.0, 5484 x 2560 x 1536 34.7 -> 29.9, 1335 x 1088 x 6856 25.9 -> 21.2, 1140 x 4352 x 7448 53 -> 44.5; E2M1 5466 x 5120 x 1528 40.6 -> 32.4.  Where 128 x 128 tiles
// make one round those are as fast or faster (30 problems of 170 to 240 192 x 192 tiles: 0.85 to 1.02), with more than one round of 192 x 192 ones both are
// (273 tiles: 22.9 against 15.5), and int8 gains 2 % at most.
static bool takes_192(const GemmProblem &p, int kind, int epi, int cus)
{
    if (kind == KIND_I8 || epi != EPI_PLAIN || !p.trans_b || (kind == KIND_F4 && scales_off_dwords(p, kind))) return false;
    if (p.tiles_192 >= 0) return p.tiles_192 != 0;
    auto tiles = [&](int64_t side) { return (p.T + side - 1) / side * ((p.N + side - 1) / side); };
    return p.kernel < 0 && p.group_sizes == nullptr && tiles(128) > 2 * cus && tiles(192) <= cus;
}

// The kernel that a problem runs on; one that "gemm_kernel" names has passed path_refuses().
static GemmPath path_of(const GemmProblem &p, int kind, int epi, int cus)
{
    if (takes_192(p, kind, epi, cus)) return PATH_MID192;
    return p.kernel >= 0 ? (GemmPath)p.kernel : choose_path(p, kind, epi, cus);
}

template <int KIND, int EPI, int FMT>
static int launch_family(const GemmProblem &p, hipStream_t stream)
{
    int dev = 0, cus = 0;
    CCH_HIP(hipGetDevice(&dev));
    CCH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (p.kernel >= 0) {
        const char *why = path_refuses(p, KIND, p.kernel);
        if (why) return fail(CCH_ENOSUP, "gemm_kernel %d does not take this problem (T=%d N=%d K=%d trans_b=%d: %s)", p.kernel, p.T, p.N, p.K, p.trans_b, why);
    }
    const GemmPath path = path_of(p, KIND, EPI, cus);
    switch (path) {
    case PATH_TILE_TAIL: {
        GemmProblem q = p;
        q.tail_cus = cus;
        const int rc = p.trans_b ? launch_tile_t<KIND, EPI, FMT, 1>(q, stream) : launch_tile_t<KIND, EPI, FMT, 0>(q, stream);
        if (rc != CCH_OK) return rc;
        return p.trans_b ? launch_mid_t<KIND, EPI, FMT, 1>(q, 64, 128, stream) : launch_mid_t<KIND, EPI, FMT, 0>(q, 64, 128, stream);
    }
    case PATH_MID1:
    case PATH_MID2:
    case PATH_MID3: {
        const int rows = PATH_MODEL[path].tm, cols = PATH_MODEL[path].tn;
        return p.trans_b ? launch_mid_t<KIND, EPI, FMT, 1>(p, rows, cols, stream) : launch_mid_t<KIND, EPI, FMT, 0>(p, rows, cols, stream);
    }
    case PATH_MID192: return launch_mid_t<KIND, EPI, FMT, 1>(p, 192, 192, stream);
    case PATH_STREAM4:
    case PATH_STREAM8: {
        const int waves = path == PATH_STREAM4 ? 4 : 8;
        return p.trans_b ? launch_stream_t<KIND, EPI, FMT, 1>(p, waves, stream) : launch_stream_t<KIND, EPI, FMT, 0>(p, waves, stream);
    }
    default: return p.trans_b ? launch_tile_t<KIND, EPI, FMT, 1>(p, stream) : launch_tile_t<KIND, EPI, FMT, 0>(p, stream);
    }
}

int launch_gemm_tile(const GemmProblem &p, int kind, int epi, hipStream_t stream)
{
    if (kind == KIND_I8 && epi == EPI_DEQUANT) return launch_family<KIND_I8, EPI_DEQUANT, 0>(p, stream);
    if (kind == KIND_I8 && epi == EPI_DEQUANT_SWIGLU) return launch_family<KIND_I8, EPI_DEQUANT_SWIGLU, 0>(p, stream);
    if (kind == KIND_F8 && epi == EPI_PLAIN && p.fmt == CCH_FMT_E4M3) return launch_family<KIND_F8, EPI_PLAIN, CCH_FMT_E4M3>(p, stream);
    if (kind == KIND_F8 && epi == EPI_PLAIN && p.fmt == CCH_FMT_E5M2) return launch_family<KIND_F8, EPI_PLAIN, CCH_FMT_E5M2>(p, stream);
    if (kind == KIND_F4 && epi == EPI_PLAIN) return launch_family<KIND_F4, EPI_PLAIN, CCH_FMT_E2M1>(p, stream);
    if (kind == KIND_F8 && epi == EPI_SWIGLU && p.fmt == CCH_FMT_E4M3) return launch_family<KIND_F8, EPI_SWIGLU, CCH_FMT_E4M3>(p, stream);
    if (kind == KIND_F8 && epi == EPI_SWIGLU && p.fmt == CCH_FMT_E5M2) return launch_family<KIND_F8, EPI_SWIGLU, CCH_FMT_E5M2>(p, stream);
    if (kind == KIND_F4 && epi == EPI_SWIGLU) return launch_family<KIND_F4, EPI_SWIGLU, CCH_FMT_E2M1>(p, stream);
    return fail(CCH_ENOSUP, "no tiled GEMM kernel for kind %d with epilogue %d, trans_b %d", kind, epi, p.trans_b);
}

}  // namespace cch

namespace cch {
// What the second launch of a grouped problem takes (gemm_tail.h), as both launches work it out: one wave.
template <bool SWIGLU>
__global__ __launch_bounds__(64) void tail_rows_kernel(GemmProblem p, int32_t *__restrict__ taken)
{
    const GroupRows rows = group_rows(p);
    const uint32_t key = tail_key<SWIGLU>(p, rows);
#pragma unroll
    for (int b = 0; b < GroupRows::NB; b++) {
        const int g = b * 64 + (int)threadIdx.x;
        if (g < p.num_groups) taken[g] = in_tail(rows, b, key) ? (rows.hi[b] - rows.lo[b]) & (BM - 1) : 0;
    }
}
}  // namespace cch

extern "C" int cch_gemm_tail_rows(const int32_t *group_sizes, int64_t num_experts, int64_t t, int64_t n, int swiglu, int cus, int32_t *taken, void *stream)
{
    using namespace cch;
    clear_error();
    CCH_REQUIRE(num_experts >= 1 && num_experts <= MAX_GROUPS, "cch_gemm_tail_rows: num_experts=%lld outside 1..%d", (long long)num_experts, MAX_GROUPS);
    CCH_REQUIRE(t >= 0 && !(t >> 31) && n >= 1 && !(n >> 31) && cus >= 1 && !(swiglu && n % 2), "cch_gemm_tail_rows: bad shape");
    CCH_REQUIRE(group_sizes && taken, "cch_gemm_tail_rows: null pointer");
    GemmProblem p{};
    p.group_sizes = group_sizes;
    p.num_groups = (int)num_experts;
    p.T = (int)t;
    p.n_out = (int)(swiglu ? n / 2 : n);
    p.tail_cus = cus;
    hipLaunchKernelGGL(swiglu ? tail_rows_kernel<true> : tail_rows_kernel<false>, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), p, taken);
    return launch_status("tail_rows_kernel");
}

extern "C" int cch_gemm_kernel_for(int fmt, int swiglu, int64_t num_experts, int64_t t, int64_t n, int64_t k, int trans_b, int cus)
{
    using namespace cch;
    if (t < 1 || n < 1 || k < 1 || t >> 31 || n >> 31 || k >> 31 || num_experts < 0 || num_experts > MAX_GROUPS || cus < 1 || (swiglu && n % 2)) return -1;
    static const int32_t some_sizes = 0;
    alignas(16) static const uint8_t some_bytes[16] = {};
    const int kind = fmt < 0 ? KIND_I8 : fmt == CCH_FMT_E2M1 ? KIND_F4 : KIND_F8, epi = kind == KIND_I8 ? (swiglu ? EPI_DEQUANT_SWIGLU : EPI_DEQUANT) : (swiglu ? EPI_SWIGLU : EPI_PLAIN);
    GemmProblem p{};
    p.a = p.b = p.sa = p.sb = some_bytes;
    p.group_sizes = num_experts > 0 ? &some_sizes : nullptr;
    p.num_groups = num_experts > 0 ? (int)num_experts : 1;
    p.T = (int)t;
    p.N = (int)n;
    p.n_out = (int)(swiglu ? n / 2 : n);
    p.K = (int)k;
    p.trans_b = trans_b;
    p.sld = kind == KIND_I8 ? 0 : (int)(2 * ((k + 63) / 64));
    p.b_stride = n * k / (kind == KIND_F4 ? 2 : 1);
    p.sb_stride = n * p.sld;
    p.kernel = p.tiles_192 = -1;
    return gemm_tile_unsupported(p, kind, epi) ? -1 : (int)path_of(p, kind, epi, cus);
}
