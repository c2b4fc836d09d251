// Host check of the workgroup -> (tensor, block) mapping that the kernels use.
//
// For random tensor lists this program builds plans with the library's own
// planner (tftq_plan.cpp, linked in), walks every workgroup id of the launch
// grid through a host restatement of the kernels' lookup (inline tables: the
// per-XCD dealt rows; device tables: chunk dealing, bucket map, binary search,
// and for reduce the quarters of workgroups that its wavefronts take one each)
// and checks that every block of every tensor is visited exactly once, in all
// three stages and in quantize's second launch.  Prints "ok <plans> plans" on success.

#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <vector>

#include "../include/tftq.h"
#include "../torchft_amd/csrc/tftq_internal.h"

static uint64_t rng_state = 0x9E3779B97F4A7C15ull;
static uint32_t rnd()
{
    rng_state ^= rng_state << 13;
    rng_state ^= rng_state >> 7;
    rng_state ^= rng_state << 17;
    return (uint32_t)(rng_state >> 32);
}

// (segment, workgroup number) of workgroup id b, or false when b has no work
static bool locate_inline(const tftq_plan *p, int st, uint32_t b, int *seg, int *vb)
{
    const int x = (int)(b & 7), i = p->natural[st] ? (int)b : (int)(b >> 3);
    const Dealt &d = p->dealt[st];
    int base = d.base[x][0], sg = d.seg[x][0];
    for (int j = 1; j < TFTQ_N_INLINE; j++)
        if (i >= d.cum_end[x][j - 1]) {
            base = d.base[x][j];
            sg = d.seg[x][j];
        }
    if (sg < 0 || i >= d.cum_end[x][TFTQ_N_INLINE - 1]) return false;
    *seg = sg;
    *vb = base + i;
    return true;
}

// wave: the wavefront of the workgroup (stages that number quarters of workgroups: reduce)
static bool locate_table(const tftq_plan *p, int st, uint32_t b, int wave, int *seg, int *vb, size_t *max_steps)
{
    const int x = (int)(b & 7), i = (int)(b >> 3);
    const int cs = p->index[st].chunk_shift;
    int v = ((((i >> cs) << 3) + x) << cs) + (i & ((1 << cs) - 1));
    if (v >= p->nwg[st]) return false;
    if (p->index[st].pieces) {
        v = 4 * v + wave;
        if (v >= p->index[st].pieces) return false;
    }
    const uint8_t *tab = p->blob.data();
    const size_t map_idx = (size_t)(v >> p->index[st].shift);
    const size_t map_bytes = (size_t)p->index[st].map_off + (map_idx + 2) * sizeof(MapEnt);
    if (map_bytes > p->blob.size()) {
        printf("map read past the table: stage %d wg %d\n", st, v);
        exit(1);
    }
    const MapEnt *m = (const MapEnt *)(tab + p->index[st].map_off) + map_idx;
    int lo = m[0].pos, sg = m[0].seg, hi = m[1].pos;
    if (lo < 0 || hi >= p->nseg || lo > hi) {
        printf("bad map entry: stage %d wg %d lo %d hi %d\n", st, v, lo, hi);
        exit(1);
    }
    if (lo != hi) {
        const SortEnt *sorted = (const SortEnt *)(tab + p->index[st].sorted_off);
        size_t steps = 0;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (sorted[mid].begin <= v) lo = mid; else hi = mid - 1;
            steps++;
        }
        if (steps > *max_steps) *max_steps = steps;
        sg = sorted[lo].seg;
    }
    *seg = sg;
    *vb = v;
    return true;
}

// by_columns: 0: contiguous rows, 1: every tensor stored column by column, 2: every other one
static int check_plan(const std::vector<int64_t> &shapes, int ws, int dtype, int by_columns = 0)
{
    const int n = (int)shapes.size() / 2;
    std::vector<int64_t> strides((size_t)n * 2);
    for (int i = 0; i < n; i++) {
        const bool cols = by_columns == 1 || (by_columns == 2 && i % 2);
        strides[2 * (size_t)i] = cols ? 1 : shapes[2 * (size_t)i + 1];
        strides[2 * (size_t)i + 1] = cols ? shapes[2 * (size_t)i] : 1;
    }
    tftq_plan *p = nullptr;
    const int rc = tftq_plan_create(dtype, n, shapes.data(), strides.data(), ws, &p);
    if (rc) {
        printf("plan_create failed: %d\n", rc);
        return 1;
    }
    const bool inl = n <= TFTQ_N_INLINE;
    if (!inl) {  // the table image starts with the descriptors in list order
        if (p->blob.size() != (size_t)tftq_plan_table_bytes(p) || tftq_plan_table_host(p) != p->blob.data() ||
            memcmp(p->blob.data(), p->segs.data(), (size_t)n * sizeof(Seg)) != 0) {
            printf("table image mismatch\n");
            return 1;
        }
    }
    for (int st = 0; st < N_LAUNCHES; st++) {
        if (st == ST_QC && p->nwg[st] == 0) continue;
        const int field = st == ST_QC ? ST_Q : st;
        // blocks each segment must receive: workgroups, or quarters of workgroups (pieces)
        const bool pieces = !inl && p->index[st].pieces > 0;
        if (pieces != (!inl && st == ST_R)) {
            printf("stage %d: pieces %d\n", st, (int)pieces);
            return 1;
        }
        std::vector<std::vector<uint8_t>> seen((size_t)n);
        int64_t total = 0;
        for (int i = 0; i < n; i++) {
            const Seg &s = p->segs[(size_t)i];
            const int64_t m_pad = (int64_t)s.slice_rows * ws;
            const int64_t rows = field == ST_Q ? m_pad : st == ST_R ? s.slice_rows : s.m;
            const int per_wg = tftq_rows_per_wg(s, field, dtype == TFTQ_F32 ? 4 : 2, ws);
            int64_t blocks = (rows + per_wg - 1) / per_wg;
            if (field == ST_Q && (s.kind[ST_Q] == K_COLS) != (st == ST_QC)) blocks = 0;  // the other launch's
            else if (st == ST_QC) blocks = (int64_t)ws * ((s.slice_rows + per_wg - 1) / per_wg);
            if (st == ST_D) {  // long rows of dequantize are dealt to several workgroups
                const int epv = dtype == TFTQ_F32 ? 4 : 8;
                const int nvec = s.n / epv;
                const int parts = s.kind[ST_D] == K_VEC256 && nvec >= 1536 ? (nvec + 1023) / 1024 : 1;
                bool ok = parts == tftq_d_row_parts(s.kind[ST_D], s.n, 16 / epv) && tftq_d_part_begin(nvec, parts, 0) == 0 &&
                          tftq_d_part_begin(nvec, parts, parts) == nvec;
                for (int k = 0; k < parts && ok && parts > 1; k++) {  // parts in order, none empty, none longer than a step
                    const int a = tftq_d_part_begin(nvec, parts, k), b = tftq_d_part_begin(nvec, parts, k + 1);
                    ok = a < b && b - a <= 1024 + 3 && (a & 3) == 0;
                }
                if (!ok) {
                    printf("segment %d: %d parts for %d vectors\n", i, parts, nvec);
                    return 1;
                }
                blocks *= s.kind[ST_D] == K_TILE ? (s.n + TFTQ_TILE_COLS - 1) / TFTQ_TILE_COLS : parts;
            }
            if (pieces) {
                blocks = tftq_reduce_pieces(s, dtype == TFTQ_F32 ? 4 : 2, ws, blocks);
                // every row of the tensor lies in one of its pieces
                const bool whole = s.kind[st] == K_GEN256 || s.kind[st] == K_COL1;
                if (whole ? blocks * per_wg < 4 * rows : blocks * (per_wg / 4) < rows || (blocks - 1) * (per_wg / 4) >= rows + (rows == 0)) {
                    printf("stage %d segment %d: %lld pieces for %lld rows\n", st, i, (long long)blocks, (long long)rows);
                    return 1;
                }
                if (tftq_reduce_kind_has_barriers(s.kind[st]) && (s.wg_begin[st] & 3)) {
                    printf("stage %d segment %d: a kind with barriers starts at piece %d\n", st, i, s.wg_begin[st]);
                    return 1;
                }
            }
            seen[(size_t)i].assign((size_t)blocks, 0);
            total += blocks;
        }
        const int64_t launched = pieces ? 4 * (int64_t)p->nwg[st] : p->nwg[st];
        if (pieces ? (total > p->index[st].pieces || p->index[st].pieces > launched || launched > p->index[st].pieces + 3)
                   : total != p->nwg[st]) {
            printf("stage %d: %lld blocks but nwg %d\n", st, (long long)total, p->nwg[st]);
            return 1;
        }
        const int64_t per_xcd = inl ? p->dealt_per_xcd[st] : p->index[st].per_xcd;
        const int64_t grid = 8 * per_xcd;
        const int64_t wgs_needed = p->nwg[st];
        const int64_t slack = inl ? 8 * n : ((int64_t)8 << p->index[st].chunk_shift) + wgs_needed / 32;
        if (grid < wgs_needed || grid > wgs_needed + slack) {
            printf("stage %d: grid %lld for %lld workgroups\n", st, (long long)grid, (long long)wgs_needed);
            return 1;
        }
        int64_t visited = 0;
        size_t max_steps = 0;
        for (int64_t b = 0; b < grid; b++) {
            for (int wave = 0; wave < (pieces ? 4 : 1); wave++) {
                int sg = -1, vb = -1;
                const bool ok = inl ? locate_inline(p, st, (uint32_t)b, &sg, &vb)
                                    : locate_table(p, st, (uint32_t)b, wave, &sg, &vb, &max_steps);
                if (!ok) continue;
                if (sg < 0 || sg >= n) {
                    printf("stage %d id %lld: segment %d\n", st, (long long)b, sg);
                    return 1;
                }
                const int64_t blk = (int64_t)vb - p->segs[(size_t)sg].wg_begin[field];
                if (pieces && blk >= (int64_t)seen[(size_t)sg].size()) {
                    // padding in front of a tensor whose kind needs whole workgroups: it must
                    // fall to a kind whose wavefronts simply find no row, of a tensor that has
                    // rows (a lane without a row of its own reads the tensor's last one)
                    if (blk >= 0 && !tftq_reduce_kind_has_barriers(p->segs[(size_t)sg].kind[st]) && blk < (int64_t)seen[(size_t)sg].size() + 3 &&
                        p->segs[(size_t)sg].slice_rows > 0)
                        continue;
                }
                if (blk < 0 || blk >= (int64_t)seen[(size_t)sg].size() || seen[(size_t)sg][(size_t)blk]) {
                    printf("stage %d id %lld: segment %d block %lld out of range or visited twice\n", st,
                           (long long)b, sg, (long long)blk);
                    return 1;
                }
                if (pieces && tftq_reduce_kind_has_barriers(p->segs[(size_t)sg].kind[st]) && (blk & 3) != wave) {
                    printf("stage %d id %lld: a workgroup of a kind with barriers is split\n", st, (long long)b);
                    return 1;
                }
                seen[(size_t)sg][(size_t)blk] = 1;
                visited++;
            }
        }
        if (visited != total) {
            printf("stage %d: visited %lld of %lld\n", st, (long long)visited, (long long)total);
            return 1;
        }
        if (max_steps > 16) {
            printf("stage %d: %zu search steps\n", st, max_steps);
            return 1;
        }
    }
    tftq_plan_destroy(p);
    return 0;
}

// The kinds that quantize and dequantize give `count` tensors of m rows and n columns stored column by
// column, behind one [4096, 4096] stored by rows if `others`.
static int check_kinds(int count, int64_t m, int64_t n, int dtype, int ws, bool others, bool cols, bool tile)
{
    std::vector<int64_t> shapes, strides;
    if (others) {
        shapes = {4096, 4096};
        strides = {4096, 1};
    }
    for (int i = 0; i < count; i++) {
        shapes.insert(shapes.end(), {m, n});
        strides.insert(strides.end(), {1, m});
    }
    tftq_plan *p = nullptr;
    if (tftq_plan_create(dtype, count + others, shapes.data(), strides.data(), ws, &p)) {
        printf("plan_create failed\n");
        return 1;
    }
    const Seg &s = p->segs.back();
    const bool ok = (s.kind[ST_Q] == K_COLS) == cols && (s.kind[ST_D] == K_TILE) == tile && (p->nwg[ST_QC] > 0) == cols;
    if (!ok)
        printf("%d x [%d, %d] dtype %d ws %d others %d: kinds %d and %d\n", count, (int)m, (int)n, dtype, ws, others, s.kind[ST_Q], s.kind[ST_D]);
    tftq_plan_destroy(p);
    return !ok;
}

int main()
{
    int plans = 0;
    // rows side by side in reduce only where enough workgroups are left
    const struct { int n, ws; int64_t rows; int at_once; } side[] = {
        {64, 2, 23000, 1}, {65, 2, 49151, 1}, {65, 2, 49152, 4}, {512, 1, 8191, 1}, {512, 1, 8192, 4}, {512, 2, 4000, 1},
        {32, 1, 262143, 1}, {32, 1, 262144, 4}, {32, 2, 1 << 22, 1}, {17, 2, 1 << 19, 1}, {17, 2, 1 << 20, 4},
        {60, 2, 1 << 19, 1}, {60, 2, 1 << 20, 4}, {46, 2, 131071, 1}, {46, 2, 131072, 4}, {65, 3, 1 << 20, 1}, {13, 2, 1 << 22, 1}};
    for (const auto &c : side) {
        const int64_t shape[] = {c.rows * c.ws, c.n}, stride[] = {c.n, 1};
        tftq_plan *p = nullptr;
        if (tftq_plan_create(TFTQ_BF16, 1, shape, stride, c.ws, &p)) return 1;
        const int got = p->segs[0].side;
        tftq_plan_destroy(p);
        if (got != c.at_once) {
            printf("%lld rows of %d columns in each of %d slots: %d rows side by side\n", (long long)c.rows, c.n, c.ws, got);
            return 1;
        }
    }
    // reduce's teams: what the whole list has to do decides, not the rows of one tensor.  Lists of `count`
    // tensors of `rows` rows per slot behind `other` of 4096 columns
    const struct { int count, rows, n, ws, other; uint8_t kind; } teams[] = {
        {1, 256, 2048, 8, 0, K_GEN256}, {1, 512, 2048, 8, 0, K_GEN64}, {2, 256, 2048, 8, 0, K_GEN64}, {44, 256, 2048, 8, 0, K_GEN64},
        {1, 256, 2048, 8, 128, K_GEN256}, {1, 256, 2048, 8, 129, K_GEN64}, {1, 511, 2048, 16, 0, K_GEN256}, {8, 511, 2048, 16, 0, K_GEN64},
        {1, 256, 1536, 64, 0, K_GEN256}, {3, 256, 1536, 64, 0, K_GEN64}, {44, 256, 2048, 4, 0, K_GEN64},
        {1, 8191, 640, 8, 0, K_GEN64}, {4, 1024, 640, 8, 0, K_GEN64}, {8, 1024, 640, 8, 0, K_GEN16}, {5, 1024, 640, 5, 0, K_GEN16}, {4, 1024, 640, 5, 0, K_GEN64}, {24, 512, 640, 4, 0, K_GEN16}, {24, 511, 640, 4, 0, K_GEN64},
        {24, 1024, 704, 8, 0, K_GEN16}, {24, 1024, 705, 8, 0, K_GEN64}, {24, 1024, 768, 7, 0, K_GEN16},
        {1, 698, 2560, 8, 0, K_GEN256}, {24, 698, 2560, 8, 0, K_GEN64}, {24, 511, 2560, 8, 0, K_GEN256}, {2, 640, 3000, 16, 0, K_GEN64}};
    for (const auto &c : teams) {
        std::vector<int64_t> shapes, strides;
        if (c.other) {
            shapes = {(int64_t)c.other * c.ws, 4096};
            strides = {4096, 1};
        }
        for (int i = 0; i < c.count; i++) {
            shapes.insert(shapes.end(), {(int64_t)c.rows * c.ws, c.n});
            strides.insert(strides.end(), {c.n, 1});
        }
        tftq_plan *p = nullptr;
        if (tftq_plan_create(TFTQ_BF16, (int)shapes.size() / 2, shapes.data(), strides.data(), c.ws, &p)) return 1;
        const int got = p->segs.back().kind[ST_R];
        tftq_plan_destroy(p);
        if (got != c.kind) {
            printf("%d x %d rows of %d columns in each of %d slots behind %d: kind %d, not %d\n", c.count, c.rows, c.n, c.ws, c.other, got, c.kind);
            return 1;
        }
    }
    // which transposed tensors are worth blocks of columns: the faster side of measured pairs
    if (check_kinds(1, 4096, 14336, TFTQ_BF16, 8, false, true, true) || check_kinds(1, 1024, 4096, TFTQ_BF16, 8, false, true, true) ||
        check_kinds(1, 256, 8192, TFTQ_BF16, 16, true, true, true) || check_kinds(1, 4096, 4096, TFTQ_F32, 64, true, true, true) ||
        check_kinds(1, 1024, 128, TFTQ_BF16, 8, false, true, true) || check_kinds(100, 1024, 256, TFTQ_F32, 16, false, true, true) ||
        check_kinds(10000, 32, 32, TFTQ_BF16, 16, false, false, false) || check_kinds(10000, 32, 32, TFTQ_F32, 2, false, false, false) ||
        check_kinds(1, 100000, 32, TFTQ_F32, 8, false, false, true) || check_kinds(1000, 128, 128, TFTQ_BF16, 64, false, false, true) ||
        check_kinds(1000, 64, 256, TFTQ_BF16, 64, false, false, true) || check_kinds(1, 64, 64, TFTQ_BF16, 8, true, false, false) ||
        check_kinds(1, 256, 256, TFTQ_BF16, 8, false, false, false) || check_kinds(512, 16, 1024, TFTQ_F32, 64, true, false, true))
        return 1;
    // widths up to the widest that a layout accepts: the blocks and tiles, whose last one is counted past
    // the row's end, stay away from it
    for (int dtype = 0; dtype < 3; dtype++)
        for (const int64_t below : {8, 9, 63, 254, 255, 256, 511, 847, 1022, 1023, 1024, 2047, 4096})
            if (check_kinds(1, 16 / (dtype == TFTQ_F32 ? 4 : 2), INT32_MAX - below, dtype, 1, false, false, false) ||
                check_kinds(20, 64, INT32_MAX - below, dtype, 3, true, false, false))
                return 1;
    // hand-picked lists: the Llama-3-8B layer bucket, empty tensors, one huge and many tiny
    const int64_t llama[] = {4096, 4096, 1024, 4096, 1024, 4096, 4096, 4096, 14336, 4096,
                             14336, 4096, 4096, 14336, 4096, 1, 4096, 1};
    if (check_plan(std::vector<int64_t>(llama, llama + 18), 8, TFTQ_BF16)) return 1;
    plans++;
    {
        std::vector<int64_t> s;
        for (int i = 0; i < 40; i++) {
            s.push_back(i % 3 == 0 ? 0 : 7 * i);
            s.push_back(i % 5 == 0 ? 0 : 3 * i + 1);
        }
        if (check_plan(s, 4, TFTQ_F32)) return 1;
        plans++;
    }
    {
        std::vector<int64_t> s = {200000, 2048};
        for (int i = 0; i < 3000; i++) {
            s.push_back(1 + i % 7);
            s.push_back(1 + i % 33);
        }
        s.push_back(0);
        s.push_back(5);
        if (check_plan(s, 16, TFTQ_BF16)) return 1;
        plans++;
    }
    {   // an empty tensor whose place by weight is right before a row that needs a whole workgroup
        std::vector<int64_t> s = {0, 12, 5, 13, 5, 2100};
        for (int i = 0; i < 15; i++) {
            s.push_back(5);
            s.push_back(4);
        }
        if (check_plan(s, 8, TFTQ_BF16)) return 1;
        plans++;
    }
    for (int n = 1; n <= 40; n += 13) {  // quantize's second launch alone: nothing but transposed tensors, some empty
        std::vector<int64_t> s;
        for (int i = 0; i < n; i++) {
            s.push_back(i % 5 == 3 ? 0 : 300 + 37 * i);
            s.push_back(700 + 131 * i);
        }
        for (int ws = 1; ws <= 16; ws += 5)
            if (check_plan(s, ws, n % 3, 1)) return 1;
        plans++;
    }
    // random lists on both sides of the inline limit
    for (int it = 0; it < 300; it++) {
        const int n = 1 + (int)(rnd() % (it % 3 == 0 ? 16 : it % 3 == 1 ? 64 : 700));
        const int ws = 1 + (int)(rnd() % 17);
        std::vector<int64_t> s;
        for (int i = 0; i < n; i++) {
            const uint32_t kind = rnd() % 8;
            int64_t m, c;
            if (kind == 0) { m = rnd() % 5000; c = 1; }
            else if (kind == 1) { m = rnd() % 40; c = 1 + rnd() % 70000; }
            else if (kind == 2) { m = 0; c = rnd() % 9; }
            else { m = rnd() % 600; c = rnd() % 700; }
            s.push_back(m);
            s.push_back(c);
        }
        for (int by_columns = 0; by_columns < 3; by_columns++) {
            if (check_plan(s, ws, (int)(rnd() % 3), by_columns)) {
                printf("failed at random list %d (n=%d ws=%d by columns %d)\n", it, n, ws, by_columns);
                return 1;
            }
            plans++;
        }
    }
    printf("ok %d plans\n", plans);
    return 0;
}
