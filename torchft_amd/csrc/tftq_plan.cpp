// Host-side planner: layout arithmetic of the packed buffer and the partition
// of rows into workgroups.  No HIP calls; compiles with any C++17 compiler.
//
// The layout restates _prepare_quantize_fp8 (torchft/quantization.py:486-503)
// and the row addressing of the kernels (:108-123).  Offsets are 64-bit here;
// the reference keeps them in int32 (:514-515).

#include <limits.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <new>
#include <vector>

#include "../../include/tftq.h"
#include "tftq_internal.h"

static inline int64_t cdiv64(int64_t a, int64_t b) { return (a + b - 1) / b; }

extern "C" int tftq_version(void) { return TFTQ_VERSION; }

#ifndef TFTQ_BUILD_ID
#define TFTQ_BUILD_ID "unknown"
#endif
extern "C" const char *tftq_build_id(void) { return TFTQ_BUILD_ID; }

extern "C" const char *tftq_strerror(int code)
{
    switch (code) {
    case 0: return "success";
    case TFTQ_E_ARG: return "invalid argument";
    case TFTQ_E_DTYPE: return "Only fp32, fp16 and bf16 are supported";
    case TFTQ_E_SHAPE: return "tensor dimension out of range";
    case TFTQ_E_SIZE: return "Output size does not match";
    case TFTQ_E_NOMEM: return "out of host memory";
    case TFTQ_E_NOTABLE: return "a list of more than 16 tensors needs the device table and the pointer buffer";
    case TFTQ_E_ARCH: return "device is not gfx950";
    case TFTQ_E_TOOBIG: return "the list's descriptor table does not fit the library's fixed array";
    case TFTQ_E_BUSY: return "the library's fixed array is still in use by a call on another stream";
    default: return code > 0 ? "HIP error" : "unknown error";
    }
}

extern "C" int tftq_layout(int n_tensors, const int64_t *shapes, int ws, int64_t *slot_off,
                           int64_t *slot_size, int64_t *output_size)
{
    if (n_tensors <= 0 || !shapes || ws <= 0) return TFTQ_E_ARG;
    int64_t per_rank = 0;
    for (int i = 0; i < n_tensors; i++) {
        const int64_t m = shapes[2 * i], n = shapes[2 * i + 1];
        if (m < 0 || n < 0 || m > INT32_MAX - ws || n > INT32_MAX - 8) return TFTQ_E_SHAPE;
        const int64_t row_bytes = (cdiv64(n, 4) + 1) * 4;
        if (slot_off) slot_off[i] = per_rank;
        per_rank += cdiv64(m, ws) * row_bytes;
        if (per_rank > (INT64_MAX / 2) / ws) return TFTQ_E_SHAPE;
    }
    if (slot_size) *slot_size = per_rank;
    if (output_size) *output_size = per_rank * ws;
    return 0;
}

// Rows that need the kernel variants with more registers (tftq_internal.h).
static bool wide_quantize(const Seg &s, int esz) { return s.kind[ST_Q] == K_VEC256 && s.n / (16 / esz) > TFTQ_Q_VECS && s.m > 0; }
static bool wide_reduce(const Seg &s, int ws)
{
    return s.kind[ST_R] == K_GEN256 && s.row_bytes / 4 - 1 > TFTQ_R_DWORDS && s.m > 0 && ws <= 64;
}

static uint8_t pick_io_kind(const Seg &s, int esz)
{
    // Vector kinds: contiguous rows of at least 64 bytes.  Neither the row start nor the
    // row length needs to be a multiple of 16 bytes: gfx950 loads and stores 16-byte
    // vectors at element alignment, and a short tail is handled per element.
    const int64_t in_bytes = (int64_t)s.n * esz;
    const bool vec_ok = s.col_stride == 1 && in_bytes >= 64;
    if (s.n == 1) return K_COL1;
    const int epv = 16 / esz;
    if (s.col_stride == 1 && s.n >= epv && tftq_small_nvec(s.n, esz) <= 32)
        return K_VECS;  // short rows of at least one vector
    if (vec_ok) {
        // Team sizes measured on MI355X inside quantize -> reduce -> dequantize sequences (a
        // kernel's time depends on what ran before it, so loops over one kernel mislead):
        // 528-byte rows are fastest with 16 lanes, 1 to 4 KB rows with 32 (1000-column bf16
        // rows: 303 us per sequence against 346 us with 16 lanes), longer ones with 64.
        if (in_bytes <= 512) return K_VEC8;
        if (in_bytes <= 1024) return K_VEC16;
        if (in_bytes <= 4096) return K_VEC32;
        if (in_bytes <= 8192) return K_VEC64;
        return K_VEC256;  // longer than 32 KB: two passes inside the workgroup
    }
    if (s.n <= 16) return K_GEN1;
    if (s.n <= 128) return K_GEN8;
    return K_GEN64;
}

// Dequantize writes rows that do not start and end on 64-byte boundaries through LDS, one
// span of 256 / team rows per workgroup (dequantize_vec_rows); the team is then the largest
// whose rows fit the stage together.  Rows of more than 16 KB have few partial lines
// and keep the team of pick_io_kind, as do rows that fill their lines.
static uint8_t pick_d_kind(const Seg &s, int esz)
{
    const uint8_t k = pick_io_kind(s, esz);
    const int64_t rowb = (int64_t)s.n * esz;
    if (k != K_VEC8 && k != K_VEC16 && k != K_VEC32 && k != K_VEC64 && k != K_VEC256) return k;
    if (s.row_stride != s.n || (rowb & 63) == 0 || rowb > 16384) {
        // Written from the registers: about three to six vectors per lane (more lanes with fewer
        // vectors each cover longer runs of memory per instruction; below three the lanes have
        // too little in flight).  8 KB rows: 116.3 us with 64 lanes of 8 vectors, 110.8 us with
        // 128 of 4; 4 KB: 117.3 -> 111.3 us; 3 KB: 118.5 -> 110.9 us; 5 KB as 128 x 2.5: 105.5
        // against 102.3 us with 64 x 5; 2 KB as 64 x 2: 115.7 against 114.3 us with 32 x 4.
        // (10 KB rows: 111.9 us with 256 lanes of 2.5 vectors, 115.7 us with 128 of 5.)
        const int64_t nvec = rowb / 16;
        if (nvec > 512) return K_VEC256;
        if (nvec >= 384) return K_VEC128;
        if (nvec >= 192) return K_VEC64;
        return k;
    }
    if (rowb <= 512) return K_VEC8;
    if (rowb <= 1024) return K_VEC16;
    if (rowb <= 2048) return K_VEC32;
    if (rowb <= 4096) return K_VEC64;
    if (rowb <= 8192) return K_VEC128;
    return K_VEC256;
}

// slot_size: bytes of the list's packed rows in a slot.
static uint8_t pick_reduce_kind(const Seg &s, int ws, int64_t slot_size)
{
    // one or two 16-byte vectors of codes per lane and peer, four for the longest rows
    const int ndw = s.row_bytes / 4 - 1;
    if (s.n == 1) return K_COL1;
    // 17 to 64 bytes of codes.  A lane per row loads its row with two or four 16-byte loads that
    // lie a row apart from its neighbours'; a pair of lanes (up to 32 bytes) or a team of 4 with
    // one vector each covers 32 or 16 neighbouring rows with one load per wavefront and peer
    // and has every load of its row in flight at once (in groups of more than 16 peers, of 8 peers
    // and the next 8).  218 M bf16 elements, 8 peers, a lane per row against the team: 24 columns
    // 81.1 -> 66.7 us, 28: 89.2 -> 64.4, 32: 65.0 -> 64.4, 44: 92.1 -> 68.7, 60: 95.6 -> 64.7, 64:
    // 70.6 -> 65.0.  45 to 48 columns are three whole vectors, of which a lane alone wastes none:
    // [2097152, 48] on rotating buffers, 4, 8, 15, 16 and 24 peers: 36.5 -> 35.2 us, 32.8 -> 31.2, 38.3 ->
    // 33.6, 31.7 -> 32.7 and 39.1 -> 33.1; in a tensor of a few rows the lane alone waits 33 us for its
    // 16 peers, the team 7 us.  (In groups of 17 to 24 peers the lane alone is up to 12 % faster on
    // millions of full rows, [4194304, 32] 17 peers 40.5 against 45.1 us, [2097152, 64] 37.0 against 42.0, and
    // up to 3 times slower on all others: [2097152, 32] 24 peers 29.2 against 24.5, 3 MB of 60 columns 17
    // peers 21.8 against 7.0.)
    if (ndw > 8 && ndw <= 16) return K_GEN4;
    if (ndw > 4 && ndw <= 8) return K_GEN2;
    if (ndw <= 16) return K_GEN1;
    if (ndw <= 32) return K_GEN8;
    if (ndw <= 64) return K_GEN16;
    // Rows that would leave more than a quarter of the next team idle take three vectors per
    // lane in a team a quarter the size (the fast path of a team holds a peer's division
    // coefficients in a lane each: ws <= lanes).  2560 bf16 columns, 8 peers: 58.9 -> 48.1 us,
    // 3072: 51.6 -> 47.9, 1280: 54.2 -> 49.9, 640: 59.1 -> 53.3.  (Not below 16 lanes: 8 lanes
    // with three vectors each are slower than 32 with one, 384 columns: 62.5 against 55.5 us.)
    // (Only for tensors with rows enough to keep the machine busy: a tensor of a few rows is
    // done sooner with more lanes per row; 10 000 tensors of up to 4096 elements: 65.0 us
    // with the smaller teams, 62.8 us without.)
    // In groups of more peers it takes more rows to keep the machine busy, as a row lives longer, the
    // more so the fewer loads its lanes have in flight.  What counts is the whole list: its tensors run
    // side by side, and it makes no difference whether it has 2048 rows in one tensor or in 32 (us, one
    // tensor / 2 to 8 of 1024 or 512 rows).  128 to 192 dwords, 16 lanes against 64: packed rows of 640 columns, 4
    // peers, 2048 rows 5.5, 5.0 / 6.0, 5.6, 4096 rows 5.7, 6.1 / 6.0, 6.4; 8 peers, 4096 rows 8.6, 6.9 / 8.9, 7.4, 8192 rows
    // in 8 tensors 11.4, 11.5; 16 peers 13.5, 11.5 / 14.1, 12.0 and 19.3, 20.1.  From 8 peers on rows of more than 176
    // dwords never win with 16: 768 columns, 60000 rows in 100 tensors 71.9, 67.4, one tensor of 40000 51.8, 46.9; with 5
    // peers 640 columns at 4096 and 8192 rows 6.4, 6.6 and 8.4, 11.1.  513
    // to 768 dwords, 64 lanes against 256: 2560 columns, 8 peers, 1024 rows 8.5, 6.9 / 9.0, 7.5, 2048 rows 10.4, 11.0 /
    // 11.1, 11.5, 16752 rows in 24 tensors 62.1, 69.9; 16 peers, 1024 rows 13.5, 11.6, 2048 rows 16.8, 19.4.
    // For the same reason rows of 257 to 512 dwords, two vectors per lane in a wavefront, go to a whole
    // workgroup: 2048 columns, 8 peers, 256 rows 5.0 -> 4.0 us, 512 in 8 tensors 5.7 -> 5.6, 1024 5.9 -> 7.4, 11264
    // in 44 35.3 -> 48.5; 16 peers, 256 rows 10.4 -> 5.4, 512 in 4 tensors 11.0 -> 7.8, 1024 11.2 -> 11.2, 4096 in 16 26.4 ->
    // 33.7; 64 peers, 256 rows 32.4 -> 12.2, 1024 36.1 -> 35.7, 2048 49.0 -> 66.0; not in groups of up to 4.
    const int64_t list_rows = slot_size / s.row_bytes;  // rows of this length that the whole list is worth
    const bool many = s.slice_rows >= 512;
    if (ndw <= 128) return K_GEN32;
    if (ndw <= (ws < 8 ? 192 : 176) && ws <= 16 && many && list_rows >= (ws <= 3 ? 512 : ws == 4 ? 2048 : ws < 8 ? 5120 : 8192)) return K_GEN16;
    if (ndw <= 256) return K_GEN64;
    if (ndw <= 512 && ws >= 5 && list_rows < (ws > 12 ? 768 : 512)) return K_GEN256;
    if (ndw <= 384 && ws <= 32 && many) return K_GEN32;
    if (ndw <= 512) return K_GEN64;
    if (ndw <= 768 && ws <= 64 && many && list_rows >= (ws <= 5 ? 512 : ws <= 8 ? 1024 : 1280)) return K_GEN64;
    return K_GEN256;
}

// Tensors whose columns are contiguous in memory (transposed matrices).  Their rows have two kernels
// each way: teams of 8 or 64 lanes with an element per lane and access (K_GEN8 up to 128 columns,
// K_GEN64), or blocks of 16 to 256 (fp32: half as many) rows in quantize (K_COLS, a launch of its own) and tiles of 64
// rows and 256 columns in dequantize (K_TILE).  The blocks and tiles read and write whole pieces of
// columns, but cost the same however many rows and columns of them the tensor has (a block never
// crosses a slot), so they lose on narrow tensors and where a slot has few rows of one.
//
// What either costs, in us: a kernel takes the longest of its workgroups' latencies, or its start and the
// work of all its tensors, whichever is more.  Quantize was fitted to kernels back to back in a graph, 980
// matrices alone, 16 to 600000 rows, 17 to 24000 columns, 1 to 32 slots, both sizes of element, each with the
// teams and with every number of groups of rows that a block can have: what is chosen takes 0.6 % more than the
// best of them in the mean, and in 41 cases more than 5 % and 0.2 us more.  Dequantize was fitted to 562
// lists.  Teams against blocks in quantize, bf16: [4096, 14336] 267 against 41 us in a graph of one
// matrix, [256, 8192] 41 against 12.3, [1024, 128] 7.0 against 4.4, 10000 [32, 32] in 16 slots 26 against 644;
// teams against tiles in dequantize: [4096, 14336] 290 against 28, [256, 256] 4.0 against 5.8, 10000 [32, 32] 18
// against 22.
struct Cost {
    double latency, work;
    double start = 3.5;
    double alone() const { return std::max(latency, start + work); }
};
constexpr double COST_HIDDEN_Q = 3.6, COST_HIDDEN_D = 4.2;  // of a latency, beside other tensors in the same launch
// What a second launch of quantize, behind one for other tensors, saves of its own: [4096, 4096] by
// rows and one transposed [64, 64], 9.6 us in one launch and 12.6 in two; [1024, 1024], 15.8 and 13.4.
constexpr double COST_OVERLAP = 0.2;

// Quantize's blocks of 2^lg groups of rows.  A block's time is a fixed part per step and the bytes it
// moves at 6.2 TB/s, slower by `slow`, as far as it uses a part of a line only, and by `wide`, where two
// workgroups no longer fit a compute unit (more than 4 steps); it counts padding lanes and rows as if they
// were real.
static Cost cost_of_blocks(const Seg &s, int lg, int esz, int ws)
{
    static const struct {
        double slow[6], wide[2], step, latency[2], per_step[2], per_column, per_column_past, start;
    } FIT[2] = {  // [0]: 2 groups, [1]: more
        {{0, 1.39, 1.13, 0.813, 0.656, 0.891}, {1.22, 1.5}, 5.03e-3, {3.01, 2.93}, {0.837, 1.02}, 7.79e-4, 3.68e-3, 2.77},   // 16 bits
        {{0, 1.12, 0.962, 0.874, 0.859, 0.923}, {1.63, 1.63}, 3.43e-3, {2.52, 3.14}, {0.611, 0.515}, 3.85e-4, 3.86e-3, 2.69}};  // fp32
    const auto &f = FIT[esz == 4];
    const int rows = tftq_qc_rows(lg, esz), steps = tftq_qc_steps(s.n, lg), more = lg > 1;
    const int held = steps <= 2 ? steps : steps <= 4 ? 4 : steps <= 8 ? 8 : 12;
    double bytes = (double)rows * s.n * (esz + 1) * f.slow[lg] * (held > 4 ? f.wide[more] : 1.0);
    double latency = f.latency[more] + f.per_step[more] * held + f.per_column * s.n;
    if (steps > 12) {  // what is read twice
        bytes *= 2.0 - 12.0 / steps;
        latency += f.per_column_past * (s.n - 12288);
    }
    const double block = hypot(f.step * held, bytes / 6.2e6);
    return {latency, (double)ws * ((s.slice_rows + rows - 1) / rows) * block, f.start};
}

static Cost cost_of(const Seg &s, uint8_t kind, int st, int esz, int ws)
{
    const double m = s.m, n = s.n, padded = (double)s.slice_rows * ws;
    const bool half = esz == 2;
    if (kind == K_COLS) return cost_of_blocks(s, s.lg_groups, esz, ws);
    if (kind == K_TILE) {
        const double tiles = (double)((s.m + TFTQ_TILE_ROWS - 1) / TFTQ_TILE_ROWS) * ((s.n + TFTQ_TILE_COLS - 1) / TFTQ_TILE_COLS);
        return {4.3 + 0.006 * std::min(n, 256.0), tiles * 1.45e-3 + m * n * esz * 1.35e-7};
    }
    if (st == ST_Q)
        return kind == K_GEN64 ? half ? Cost{2.56 + 0.0052 * n, padded * n * 3.97e-6, 2.03} : Cost{2.41 + 0.00441 * n, padded * n * 5.51e-6, 1.5}
               : half          ? Cost{2.22 + 0.0288 * n, padded * (n * 1.85e-6 + 5.0e-7), 2.71}
                               : Cost{2.28 + 0.0255 * n, padded * (n * 1.94e-6 + 3.63e-6), 2.52};
    return kind == K_GEN64 ? Cost{2.9 + 0.0044 * n, m * n * 4.0e-6}
                           : Cost{3.0 + 0.021 * n, m * (n * 1.0e-6 + (half ? 1.4e-5 : 2.0e-5))};
}

static bool stored_by_columns(const Seg &s, int st, int esz)
{
    // (fp32 rows of up to 32 columns stay with their teams in quantize.)
    constexpr int MOST = INT32_MAX - 4096;  // the blocks and tiles round rows and columns up
    return s.row_stride == 1 && s.m >= 16 / esz && s.m < MOST && s.n < MOST &&
           (s.kind[st] == K_GEN8 || s.kind[st] == K_GEN64) && (st != ST_Q || esz == 2 || s.n > 32);
}

// How many groups of rows a block of quantize holds (Seg::lg_groups).  More make whole lines of what it
// reads and fewer blocks, and fewer columns per step (tftq_qc_has); more than 4 steps of more than 2
// groups (a workgroup per compute unit) are for tensors of 192 blocks: bf16 [5682, 4287] in 16 slots, say.  A
// tensor takes the groups that are the least work, or, if the launch has little else to do, those that are
// done soonest.  us in 2 / 4 / 8 / 16 / 32 groups, bf16, 8 slots:
// [2330168, 18] 920 / 458 / 232 / 126 / 65, [42799, 147] 18.5 / 11.0 / 8.0 / 7.0 / 8.1, [3495, 300] 4.7 / 4.6 / 5.8 /
// 8.3 / -, [41943, 1000] 30.4 / 25.1 / 21.9 / - / -, [1048, 1000] 5.1 / 6.3 / 9.0 / - / -, [11983, 3500] 28.9 / 34.0 / - / -
// / -, fp32 63.6 / 51.6.
static void pick_groups(tftq_plan *p)
{
    double least[2] = {0.0, 0.0};  // all tensors' work with the groups that are the least of it; one tensor's
    for (int pass = 0; pass < 2; pass++)
        for (Seg &s : p->segs) {
            if (!stored_by_columns(s, ST_Q, p->esz)) continue;
            Cost cost[6];
            int most = 1;
            for (int lg = 1; lg <= 5 && tftq_qc_has(lg, tftq_qc_steps(s.n, lg)); lg++) {
                const int rows = tftq_qc_rows(lg, p->esz);
                if (lg > 1 && tftq_qc_steps(s.n, lg) > 4 && (int64_t)p->ws * ((s.slice_rows + rows - 1) / rows) < 192) break;
                cost[lg] = cost_of_blocks(s, lg, p->esz, p->ws);
                most = lg;
            }
            least[1] = HUGE_VAL;
            for (int lg = 1; lg <= most; lg++) least[1] = std::min(least[1], cost[lg].work);
            if (pass == 0) {
                least[0] += least[1];
                continue;
            }
            double best = HUGE_VAL;
            for (int lg = 1; lg <= most; lg++) {
                const double t = std::max(cost[lg].latency, cost[lg].start + least[0] - least[1] + cost[lg].work);
                if (t >= best) continue;
                best = t;
                s.lg_groups = (uint8_t)lg;
            }
        }
}

// Chooses for a stage between the teams that the tensors have been given and `blocks` (K_COLS or
// K_TILE): for none of them, for those that it makes less work, or for all (a few tensors that the
// machine takes at once, where only the latency counts).
static void pick_column_kinds(tftq_plan *p, int st, uint8_t blocks)
{
    enum { NONE, LESS_WORK, ALL, N_WAYS };
    // per way: what is left to the teams, what goes to the blocks
    const Cost nothing = {0.0, 0.0, 0.0};
    Cost teams[N_WAYS] = {nothing, nothing, nothing}, taken[N_WAYS] = {nothing, nothing, nothing};
    bool any[N_WAYS] = {}, others = false;
    for (const Seg &s : p->segs) {
        if (!stored_by_columns(s, st, p->esz)) {
            others = others || s.m > 0;
            continue;
        }
        const Cost t = cost_of(s, s.kind[st], st, p->esz, p->ws), b = cost_of(s, blocks, st, p->esz, p->ws);
        for (int way = NONE; way < N_WAYS; way++) {
            const bool take = way == ALL || (way == LESS_WORK && b.work < t.work);
            Cost &sum = take ? taken[way] : teams[way];
            const Cost &c = take ? b : t;
            sum = {std::max(sum.latency, c.latency), sum.work + c.work, std::max(sum.start, c.start)};
            any[way] = any[way] || take;
        }
    }
    int best = NONE;
    double least = HUGE_VAL;
    for (int way = NONE; way < N_WAYS; way++) {
        auto launch = [&](const Cost &c) {
            if (others) return std::max(c.latency - (st == ST_D ? COST_HIDDEN_D : COST_HIDDEN_Q), c.work);
            return c.latency > 0.0 ? c.alone() : 0.0;
        };
        const Cost &a = teams[way], &b = taken[way];
        double t;
        if (st == ST_D) {
            t = launch({std::max(a.latency, b.latency), a.work + b.work});
        } else {
            t = launch(a);
            if (any[way]) t += b.alone() - (others ? COST_OVERLAP : 0.0);
        }
        if (t < least) {
            least = t;
            best = way;
        }
    }
    if (!any[best]) return;
    for (Seg &s : p->segs)
        if (stored_by_columns(s, st, p->esz) &&
            (best == ALL || cost_of(s, blocks, st, p->esz, p->ws).work < cost_of(s, s.kind[st], st, p->esz, p->ws).work))
            s.kind[st] = blocks;
}

// Gives every block of a list 2 groups where the tensors' own choices would gain little.  Rows of more than
// 4 steps run in a kernel of their own where all blocks of the list have 2 groups, 4 to 9 % sooner than in the
// general one (us, 8 slots: [4096, 14336] beside [4096, 1024] in 2 and in 8 groups, bf16 64.2 and 68.8, fp32 114.6
// and 125.3).  And a few small tensors are done sooner if none of them has blocks that live long: bf16
// [231, 2922] and [803, 2922] 10.8 with their own, 10.2 in 2 groups, 8 slots, [251, 224], [2344, 672] and [248, 672]
// 5.5 and 4.9, fp32 [181, 1573], [1620, 1573] and [162, 524] in one slot 8.1 and 6.7.
static void pick_two_groups(tftq_plan *p)
{
    constexpr double LOSS = 0.07, LOSS_SMALL = 0.25, SMALL = 10.0;
    double wide = 0.0;
    int64_t blocks = 0;  // in 2 groups
    Cost two = {0.0, 0.0, 0.0}, own = two;
    for (const Seg &s : p->segs) {
        if (s.kind[ST_Q] != K_COLS) continue;
        const Cost a = cost_of_blocks(s, 1, p->esz, p->ws), b = cost_of_blocks(s, s.lg_groups, p->esz, p->ws);
        two = {std::max(two.latency, a.latency), two.work + a.work, a.start};
        own = {std::max(own.latency, b.latency), own.work + b.work, b.start};
        if (s.lg_groups == 1 && tftq_qc_steps(s.n, 1) > 4) wide += a.work;
        const int rows = tftq_qc_rows(1, p->esz);
        blocks += (int64_t)p->ws * ((s.slice_rows + rows - 1) / rows);
    }
    // (in 16 bits only what the kernel for few blocks takes)
    const bool small = p->nseg > 1 && (p->esz == 4 || blocks <= 256) && two.alone() < SMALL && two.alone() < (1.0 + LOSS_SMALL) * own.alone();
    if (!small && (wide == 0.0 || two.work - own.work >= LOSS * wide)) return;
    for (Seg &s : p->segs)
        if (s.kind[ST_Q] == K_COLS) s.lg_groups = 1;
}

// Kinds for little work.  K_VECS gives a lane 8 vectors, in 2 to 8 rows one after the other, and K_COL1
// up to 8 rows (reduce: 4 rows and a peer at a time), which is what a machine full of workgroups wants;
// where there are too few to fill it, a stage takes as long as one workgroup lives, and a quarter of the
// work per lane takes half as long.  Measured with the kernels back to back, 8 peers unless said:
//   quantize, K_VECS: [630, 13] bf16 5.3 -> 3.3 us, [3449, 38] 6.8 -> 3.5, [256, 256] 5.7 -> 3.7; 8 MB of
//     [20971, 200] 7.1 -> 5.9, of fp32 [55188, 38] 7.3 -> 6.3; 16 MB of 38 to 256 columns 10.3 -> 9.8 to 8.5 ->
//     8.4, of fp32 [110376, 38] 9.4 -> 9.6; 32 MB mostly slower ([441505, 38] 14.5 -> 16.0);
//   dequantize, K_VECS: [630, 13] 5.2 -> 3.3, [3449, 38] 5.3 -> 3.6, [256, 256] 4.6 -> 3.2; 8 MB of [20971, 200]
//     7.5 -> 6.5, of fp32 [55188, 38] 6.2 -> 5.5; rows that fill their 64-byte blocks: 4 MB of [8192, 256] 5.5 ->
//     4.6, 8 MB of [16384, 256] 5.8 -> 6.0;
//   either, in long lists: a tensor whose rows are those of one workgroup of K_VECS leaves most of its lanes'
//     rows empty: 10000 tensors of up to 4096 elements, 16 peers, 48.6 -> 44.3 and 30.2 -> 27.8;
//   quantize, K_COL1: vectors of up to 4 MB, bf16 2^12 elements 3.6 -> 2.8 us, 2^21 6.9 -> 5.8, 2^22 11.4 -> 12.2
//     (not in long lists: 48.6 -> 51.0);
//   reduce, K_COL1, up to 262144 rows per slot, 2 / 4 / 8 / 16 / 64 peers: 2^17 elements 3.2 -> 2.9, 4.3 -> 3.0,
//     4.9 -> 3.2, 7.1 -> 3.4, 39.5 -> 7.0; 2 to 8 peers at 262144 rows 3.5 -> 3.4, 5.3 -> 3.8, 8.0 -> 5.9, at
//     524288 6.2 -> 7.2, 6.5 -> 6.7, 10.1 -> 10.6; more peers at 524288 rows 17.9 -> 13.8 (16), 59 -> 47 (64), at
//     1048576 24.0 -> 24.2 (16), 44.3 -> 45.7 (32); in long lists where a tensor has no more rows than a workgroup of
//     K_COL1: 20000 tensors, 8 peers, 48.9 -> 43.0 (2 peers: 28.7 -> 34.8).  Not in lists that the kernel for long
//     rows (R_LONG) takes, which holds no such code, unless they are small as a whole.
static void pick_few_kinds(tftq_plan *p)
{
    constexpr double MB = 1 << 20;
    constexpr double Q_VECS = 12 * MB, D_VECS = 8 * MB, D_VECS_FILLED = 4 * MB, Q_COL1 = 4 * MB, R_LONG_LIST = 4 * MB;
    double bytes = 0.0, vector_rows = 0.0;
    bool wide_q = false, wide_r = false, long_rows = true, vectors_only = true;
    for (const Seg &s : p->segs) {
        bytes += (double)s.m * s.n * p->esz;
        if (s.kind[ST_R] == K_COL1) vector_rows += s.slice_rows;
        else if (s.m > 0) vectors_only = false;
        if (s.m > 0 && s.kind[ST_R] != K_COL1 && s.kind[ST_R] != K_GEN64 && s.kind[ST_R] != K_GEN256) long_rows = false;
        wide_q = wide_q || wide_quantize(s, p->esz);
        wide_r = wide_r || wide_reduce(s, p->ws);
    }
    const bool few_vectors = vector_rows <= (p->ws > 8 ? 524288 : 262144);
    for (Seg &s : p->segs) {
        if (s.kind[ST_Q] == K_VECS || s.kind[ST_D] == K_VECS) {
            const int64_t per_wg = tftq_small_rows_per_wg(tftq_small_nvec(s.n, p->esz), ST_Q, TFTQ_SMALL_VECS);
            const bool filled = ((int64_t)s.n * p->esz) % 64 == 0;
            if (s.kind[ST_Q] == K_VECS && !wide_q && (bytes <= Q_VECS || (int64_t)s.slice_rows * p->ws <= per_wg))
                s.kind[ST_Q] = K_VECS_FEW;
            if (s.kind[ST_D] == K_VECS && (bytes <= (filled ? D_VECS_FILLED : D_VECS) || s.m <= per_wg)) s.kind[ST_D] = K_VECS_FEW;
        }
        if (s.kind[ST_Q] == K_COL1 && !wide_q && p->nseg <= TFTQ_N_INLINE && bytes <= Q_COL1) s.kind[ST_Q] = K_COL1_FEW;
        if (s.kind[ST_R] == K_COL1 && !wide_r && (vectors_only || !long_rows || bytes <= R_LONG_LIST) &&
            (few_vectors || (s.slice_rows <= tftq_col1_rows_per_wg(ST_R) && p->ws >= 4)))
            s.kind[ST_R] = K_COL1_FEW;
    }
}

// Bytes one workgroup of segment s moves in reduce.
static double reduce_weight(const Seg &s, int esz, int ws)
{
    return (double)tftq_rows_per_wg(s, ST_R, esz, ws) * (double)s.row_bytes * (ws + 1);
}

// The order in which a stage works through the segments.  Reduce: by workgroup
// weight, heaviest first (equal weights keep the list order), so that the last
// workgroups to finish are light; its weights differ by orders of magnitude
// within one list.  Empty tensors come before all others: the pieces that pad the numbering up to a
// whole workgroup (build_table) belong to the tensor in front of them, whose lanes without a row of
// their own read its last row, so it must have one.
// Quantize and dequantize keep the list order: their
// workgroups are all of similar weight, and sorting them measured slower.
static void work_order(const tftq_plan *p, int st, std::vector<int32_t> &ord)
{
    ord.resize((size_t)p->nseg);
    for (int i = 0; i < p->nseg; i++) ord[(size_t)i] = i;
    if (st != ST_R) return;
    std::vector<double> w((size_t)p->nseg);
    for (int i = 0; i < p->nseg; i++) {
        const Seg &s = p->segs[(size_t)i];
        w[(size_t)i] = s.m > 0 ? reduce_weight(s, p->esz, p->ws) : HUGE_VAL;
    }
    std::stable_sort(ord.begin(), ord.end(), [&](int32_t a, int32_t b) { return w[(size_t)a] > w[(size_t)b]; });
}

// Whether a stage hands its workgroups to the XCDs in their natural order (workgroup id b is
// piece b of the work: neighbouring pieces run on different XCDs at the same time and the
// whole chip works on one compact window of memory) instead of a contiguous eighth per XCD.
// Measured on MI355X, kernel sequences on 218 M elements: dequantize is 1 to 6 % faster in
// natural order (4096 bf16 columns 122.0 -> 117.9 us, 14336: 122.4 -> 115.7, 256: 148.0 ->
// 140.4, 4096 fp32: 101.4 -> 96.3) when the tensor rows are whole 64-byte blocks, and 5 %
// slower when they are not (1000 columns: neighbouring rows then share blocks across XCDs);
// quantize, which writes its packed rows as whole lines from LDS, gains 2 % (benchmark
// configuration 3: 114.0 -> 111.6 us); reduce does not care and keeps the eighths, which
// its heaviest-first order is built on.
static bool natural_order(const tftq_plan *p, int st)
{
    if (st == ST_R || st == ST_QC) return false;
    double whole = 0.0, all = 0.0;
    for (int i = 0; i < p->nseg; i++) {
        const Seg &s = p->segs[(size_t)i];
        const double bytes = (double)s.m * (double)s.n * p->esz;
        const bool fills = s.n == 1 ? s.row_stride == 1
                                    : s.col_stride == 1 && ((int64_t)s.n * p->esz) % 64 == 0 &&
                                          (s.row_stride * p->esz) % 64 == 0;
        all += bytes;
        if (fills) whole += bytes;
    }
    return whole * 2.0 >= all && all > 0.0;
}

// Few segments (the table travels in the kernel arguments).  Workgroup ids are
// dealt round-robin to the 8 XCDs by the hardware; here every XCD takes a
// contiguous eighth of every segment, so all XCDs see the same mix of row
// lengths, and works through the segments in work_order().
static void deal_to_xcds(tftq_plan *p, const int32_t (*wgs)[N_LAUNCHES])
{
    for (int st = 0; st < N_LAUNCHES; st++) {
        const int field = st == ST_QC ? ST_Q : st;
        int32_t begin = 0;
        for (int i = 0; i < p->nseg; i++) {  // workgroup numbers in list order
            if (st == ST_QC && wgs[i][st] == 0) continue;  // numbered for ST_Q
            p->segs[(size_t)i].wg_begin[field] = begin;
            begin += wgs[i][st];
        }
        std::vector<int32_t> ord;
        work_order(p, st, ord);
        Dealt &d = p->dealt[st];
        int64_t busiest = 0;
        p->natural[st] = natural_order(p, st);
        for (int x = 0; x < 8; x++) {
            int64_t cum = 0;
            for (int k = 0; k < TFTQ_N_INLINE; k++) {
                if (k >= p->nseg) {
                    d.cum_end[x][k] = INT32_MAX;
                    d.base[x][k] = 0;
                    d.seg[x][k] = -1;
                    continue;
                }
                const int i = ord[(size_t)k];
                const uint64_t n = (uint64_t)wgs[i][st];
                // natural order: every row of the table covers all workgroups of every segment
                const int64_t lo = p->natural[st] ? 0 : (int64_t)((n * (uint64_t)x) >> 3);
                const int64_t hi = p->natural[st] ? (int64_t)n : (int64_t)((n * (uint64_t)(x + 1)) >> 3);
                d.base[x][k] = (int32_t)(p->segs[(size_t)i].wg_begin[field] + lo - cum);
                d.seg[x][k] = i;
                cum += hi - lo;
                d.cum_end[x][k] = (int32_t)cum;
            }
            if (cum > busiest) busiest = cum;
        }
        p->dealt_per_xcd[st] = (int32_t)(p->natural[st] ? (busiest + 7) / 8 : busiest);
    }
}

// Many segments: the image of the device table (layout in tftq_internal.h).
static int build_table(tftq_plan *p, const int32_t (*wgs)[N_LAUNCHES])
{
    const size_t nseg = (size_t)p->nseg;
    std::vector<SortEnt> sorted[N_LAUNCHES];
    std::vector<MapEnt> map[N_LAUNCHES];
    const int launches = p->nwg[ST_QC] ? N_LAUNCHES : 3;  // no index for a launch that no tensor needs
    for (int st = 0; st < launches; st++) {
        std::vector<int32_t> ord;
        work_order(p, st, ord);
        sorted[st].resize(nseg);
        // Reduce numbers quarters of workgroups (tftq_reduce_pieces), the others whole workgroups.
        const bool pieces = st == ST_R;
        int64_t begin = 0;
        for (size_t k = 0; k < nseg; k++) {  // workgroup (piece) numbers in sorted order
            const int32_t i = ord[k];
            const Seg &sg = p->segs[(size_t)i];
            if (pieces && tftq_reduce_kind_has_barriers(sg.kind[st])) begin = (begin + 3) & ~(int64_t)3;
            if (begin > INT32_MAX - 4096) return TFTQ_E_SHAPE;
            if (st != ST_QC) p->segs[(size_t)i].wg_begin[st] = (int32_t)begin;
            else if (wgs[i][st]) p->segs[(size_t)i].wg_begin[ST_Q] = (int32_t)begin;
            sorted[st][k] = SortEnt{(int32_t)begin, i};
            begin += pieces ? tftq_reduce_pieces(sg, p->esz, p->ws, wgs[i][st]) : wgs[i][st];
        }
        if (begin > INT32_MAX - 4096) return TFTQ_E_SHAPE;
        p->index[st].pieces = pieces ? (int32_t)begin : 0;
        if (pieces) p->nwg[st] = (int32_t)((begin + 3) / 4);
        const int64_t nwg = begin;  // what the map is indexed by
        int shift = 0;
        while ((nwg >> shift) > 4 * (int64_t)nseg) shift++;
        const int64_t nb = (nwg >> shift) + 1;  // buckets; map[] has one more entry
        map[st].resize((size_t)nb + 1);
        size_t k = 0;
        for (int64_t b = 0; b <= nb; b++) {
            const int64_t w = b << shift;
            if (w >= nwg) {
                k = nseg - 1;
            } else {
                while (k + 1 < nseg && sorted[st][k + 1].begin <= w) k++;
            }
            map[st][(size_t)b] = MapEnt{(int32_t)k, sorted[st][k].seg};
        }
        p->index[st].shift = shift;
        const int64_t nwgs = p->nwg[st];  // workgroups of the launch
        int cs = 4;
        while (cs < 20 && (nwgs >> (cs + 1)) >= 8 * 64) cs++;
        p->index[st].chunk_shift = cs;
        const int64_t turns = (nwgs + ((int64_t)8 << cs) - 1) / ((int64_t)8 << cs);
        p->index[st].per_xcd = (int32_t)(turns << cs);
    }
    size_t bytes = nseg * sizeof(Seg);
    auto place = [&](int begin, int end) {
        for (int st = begin; st < end; st++) {
            p->index[st].sorted_off = (int64_t)bytes;
            bytes += nseg * sizeof(SortEnt);
        }
        for (int st = begin; st < end; st++) {
            p->index[st].map_off = (int64_t)bytes;
            bytes += map[st].size() * sizeof(MapEnt);
        }
    };
    place(0, 3);
    p->static_bytes = bytes;
    place(3, launches);  // quantize's second launch, last: tftq_reduce_static leaves it out
    p->blob.resize(bytes);
    memcpy(p->blob.data(), p->segs.data(), nseg * sizeof(Seg));
    for (int st = 0; st < launches; st++) {
        memcpy(p->blob.data() + p->index[st].sorted_off, sorted[st].data(), nseg * sizeof(SortEnt));
        memcpy(p->blob.data() + p->index[st].map_off, map[st].data(), map[st].size() * sizeof(MapEnt));
    }
    return 0;
}

extern "C" int tftq_plan_create(int dtype, int n_tensors, const int64_t *shapes, const int64_t *strides,
                                int ws, tftq_plan **out)
{
    if (!out) return TFTQ_E_ARG;
    *out = nullptr;
    if (dtype != TFTQ_F32 && dtype != TFTQ_F16 && dtype != TFTQ_BF16) return TFTQ_E_DTYPE;
    if (n_tensors <= 0 || !shapes || !strides || ws <= 0) return TFTQ_E_ARG;

    tftq_plan *p = new (std::nothrow) tftq_plan();
    if (!p) return TFTQ_E_NOMEM;
    p->dtype = dtype;
    p->esz = dtype == TFTQ_F32 ? 4 : 2;
    p->ws = ws;
    p->nseg = n_tensors;
    p->max_rows = 0;
    std::vector<int64_t> offs;
    std::vector<int32_t> wgs_flat;
    try {  // nothing may throw across the C ABI
        p->segs.resize((size_t)n_tensors);
        offs.resize((size_t)n_tensors);
        wgs_flat.resize((size_t)n_tensors * N_LAUNCHES);
    } catch (...) {
        delete p;
        return TFTQ_E_NOMEM;
    }
    int rc = tftq_layout(n_tensors, shapes, ws, offs.data(), &p->slot_size, &p->output_size);
    if (rc) {
        delete p;
        return rc;
    }
    p->cols_two = true;
    int64_t wg[N_LAUNCHES] = {0, 0, 0, 0};
    int32_t (*wgs)[N_LAUNCHES] = (int32_t (*)[N_LAUNCHES])wgs_flat.data();  // workgroups per segment and launch
    for (int i = 0; i < n_tensors; i++) {
        Seg &s = p->segs[(size_t)i];
        memset(&s, 0, sizeof(s));
        s.ptr = 0;
        s.slot_off = offs[(size_t)i];
        s.m = (int32_t)shapes[2 * i];
        s.n = (int32_t)shapes[2 * i + 1];
        s.row_stride = strides[2 * i];
        s.col_stride = strides[2 * i + 1];
        s.slice_rows = (int32_t)cdiv64(s.m, ws);
        s.row_bytes = (int32_t)((cdiv64(s.n, 4) + 1) * 4);
        const int64_t m_pad = (int64_t)s.slice_rows * ws;
        if (m_pad > p->max_rows) p->max_rows = m_pad;

        s.kind[ST_Q] = pick_io_kind(s, p->esz);
        s.kind[ST_D] = pick_d_kind(s, p->esz);
        s.kind[ST_R] = pick_reduce_kind(s, p->ws, p->slot_size);
        s.side = (uint8_t)tftq_reduce_rows_side(s.kind[ST_R], s.row_bytes / 4 - 1, s.slice_rows, p->ws);
    }
    pick_few_kinds(p);
    pick_groups(p);
    pick_column_kinds(p, ST_Q, K_COLS);
    pick_two_groups(p);
    pick_column_kinds(p, ST_D, K_TILE);
    for (int i = 0; i < n_tensors; i++) {
        Seg &s = p->segs[(size_t)i];
        const int64_t rows[3] = {(int64_t)s.slice_rows * ws, s.slice_rows, s.m};
        for (int st = 0; st < 3; st++) {
            const int64_t n = tftq_wgs_of(s, st, p->esz, ws, rows[st]);
            const int launch = s.kind[st] == K_COLS ? ST_QC : st;
            wgs[i][st] = 0;
            wgs[i][launch] = (int32_t)n;
            wg[launch] += n;
            if (wg[launch] > INT32_MAX - 4096) {
                delete p;
                return TFTQ_E_SHAPE;
            }
        }
        if (s.kind[ST_Q] == K_COLS) {
            p->cols_most = std::max(p->cols_most, tftq_qc_steps(s.n, s.lg_groups));
            p->cols_two = p->cols_two && s.lg_groups == 1;
        }
    }
    for (int st = 0; st < N_LAUNCHES; st++) p->nwg[st] = (int32_t)wg[st];
    p->wide[ST_Q] = p->wide[ST_R] = p->wide[ST_D] = false;
    p->parked = 0;
    p->reduce_long_rows = p->reduce_one_column = true;
    for (int i = 0; i < n_tensors; i++) {
        const Seg &s = p->segs[(size_t)i];
        const int nvec = s.n / (16 / p->esz);
        if (s.m > 0 && s.kind[ST_R] != K_GEN256 && s.kind[ST_R] != K_GEN64 && s.kind[ST_R] != K_COL1)
            p->reduce_long_rows = false;
        if (s.m > 0 && s.kind[ST_R] != K_COL1 && s.kind[ST_R] != K_COL1_FEW) p->reduce_one_column = false;
        if (wide_quantize(s, p->esz)) p->wide[ST_Q] = true;
        if (s.kind[ST_Q] == K_VEC256 && nvec > TFTQ_Q_VECS_WIDE && s.m > 0) p->parked = std::max(p->parked, tftq_q_park_groups(nvec));
        if (wide_reduce(s, ws)) p->wide[ST_R] = true;
    }
    try {
        if (p->nseg <= TFTQ_N_INLINE) {
            deal_to_xcds(p, wgs);
        } else if (const int rc = build_table(p, wgs)) {
            delete p;
            return rc;
        }
    } catch (...) {
        delete p;
        return TFTQ_E_NOMEM;
    }
    // a grid has fewer than 2^32 threads
    for (int st = 0; st < N_LAUNCHES; st++) {
        const int64_t per_xcd = p->nseg <= TFTQ_N_INLINE ? p->dealt_per_xcd[st] : p->index[st].per_xcd;
        if (8 * per_xcd * (st == ST_QC ? TFTQ_QC_WG : TFTQ_WG) > (int64_t)UINT32_MAX) {
            delete p;
            return TFTQ_E_SHAPE;
        }
    }
    *out = p;
    return 0;
}

extern "C" void tftq_plan_destroy(tftq_plan *plan) { delete plan; }

extern "C" int64_t tftq_plan_output_size(const tftq_plan *plan) { return plan ? plan->output_size : -1; }
extern "C" int64_t tftq_plan_slot_size(const tftq_plan *plan) { return plan ? plan->slot_size : -1; }
extern "C" int64_t tftq_plan_max_rows(const tftq_plan *plan) { return plan ? plan->max_rows : -1; }
extern "C" int tftq_plan_n_tensors(const tftq_plan *plan) { return plan ? plan->nseg : -1; }

extern "C" int64_t tftq_plan_table_bytes(const tftq_plan *plan)
{
    if (!plan) return -1;
    return plan->nseg > TFTQ_N_INLINE ? (int64_t)plan->blob.size() : 0;
}

extern "C" const void *tftq_plan_table_host(const tftq_plan *plan)
{
    if (!plan) return nullptr;
    return plan->nseg > TFTQ_N_INLINE ? (const void *)plan->blob.data() : nullptr;
}
