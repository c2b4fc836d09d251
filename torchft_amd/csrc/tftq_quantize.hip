// k_quantize and tftq_quantize: fused_quantize_into_fp8 on gfx950.
//
// Follows torchft/quantization.py:53-162 (kernel) and :531-588 (launcher); design notes in tftq_device.h.

#include "tftq_device.h"

// ---------------------------------------------------------------------------
// quantize
// ---------------------------------------------------------------------------
constexpr int QV = 8;  // 16-byte vectors a lane keeps in registers

template <typename T>
DEV float vec_absmax(const u32x4 v)
{
    float f[Elem<T>::EPV];
    Elem<T>::unpack(v, f);
    float a = 0.0f;
#pragma unroll
    for (int e = 0; e < Elem<T>::EPV; e++) a = fmaxf(a, __builtin_fabsf(f[e]));
    return a;
}

// the 4 (fp32) or 8 (16-bit) codes of one input vector: one or two dwords
template <typename T>
DEV u32x2 vec_codes(const u32x4 v, float s)
{
    float f[Elem<T>::EPV];
    Elem<T>::unpack(v, f);
    u32x2 o = {0u, 0u};
    o.x = pack_fp8x4(f[0] * s, f[1] * s, f[2] * s, f[3] * s);
    if constexpr (Elem<T>::EPV == 8) o.y = pack_fp8x4(f[4] * s, f[5] * s, f[6] * s, f[7] * s);
    return o;
}

template <typename T>
DEV void vec_quant_store(const u32x4 v, float s, GLOBAL u32 *payload, int idx)
{
    const u32x2 o = vec_codes<T>(v, s);
    if constexpr (Elem<T>::EPV == 4) {
        payload[idx] = o.x;
    } else {
        *(GLOBAL u32x2_a4 *)(payload + 2 * idx) = o;  // plain store: rows start 4 bytes off a line, L2 merges
    }
}

// Lanes past the last vector of a row re-read its last vector, moved down to a 16-byte
// boundary when the row starts off one (the row has at least two vectors, so the bytes
// are still the row's): whole wavefronts of such lanes then cost one aligned access, while
// 64 copies of a vector at an odd 2-byte offset are served lane by lane (10001-column
// bf16 rows, five vectors per lane needed and eight loaded: 153.8 us against 117.1 us for 10000).
DEV int dup_vec_offset(GLOBAL const u32x4_a2 *in, int nvec)
{
    return (nvec - 1) * 16 - (int)((uintptr_t)in & 15u);
}
DEV GLOBAL const u32x4_a2 *vec_or_dup(GLOBAL const u32x4_a2 *in, int idx, int nvec, int dup)
{
    return (GLOBAL const u32x4_a2 *)((GLOBAL const uint8_t *)in + (idx < nvec ? idx * 16 : dup));
}

constexpr int Q_STAGE_BYTES = 16640;  // 8 rows of 2052 bytes (2048 16-bit columns) + 127 bytes of offset, rounded up (see copy_out_span)
// the wide kernel, whose three workgroups per CU leave each 53 KB of LDS: one row of 32768 16-bit columns
constexpr int Q_STAGE_BYTES_WIDE = 32912;

// Contiguous, 16-byte aligned rows of at most TEAM * KMAX vectors.  The KMAX
// loads of a lane are issued back to back without a branch in between: lanes
// past the end of the row re-read its last vector (a duplicate cannot change
// the maximum) and simply do not store.
// STAGED: the row is a real one and its packed image goes to LDS at srow (see copy_out_span).
template <typename T, int TEAM, int KMAX, bool STAGED = false>
DEV void quantize_vec_k(const Seg &s, const KCall &p, int row, int lane, float *lds, LDS_AS u32 *srow = nullptr)
{
    GLOBAL u32 *out = nullptr;
    if (!STAGED) {
        const bool active = row < s.slice_rows * p.ws;
        out = as_global<u32>(p.packed + (active ? row_addr(s, p.slot_size, row) : 0));
        if (active && row >= s.m) {
            // padding row: the reference leaves it zero (:93-95 on a zero-filled buffer)
            for (int d = lane; d < (s.row_bytes >> 2); d += TEAM) out[d] = 0;
        }
        if (!active || row >= s.m) return;  // a team leaves whole: its lanes share the row
    }

    constexpr int EPV = Elem<T>::EPV;
    const int nvec = s.n / EPV;
    const int tail = s.n - nvec * EPV;  // elements after the last whole vector (rare)
    const int64_t r0 = (int64_t)row * s.row_stride;
    GLOBAL const u32x4_a2 *in = as_global<const u32x4_a2>(s.ptr + r0 * Elem<T>::ESZ);
    const int dup = dup_vec_offset(in, nvec);
    u32x4 v[KMAX];
#pragma unroll
    for (int k = 0; k < KMAX; k++) v[k] = LOAD_STREAM(vec_or_dup(in, k * TEAM + lane, nvec, dup));
    // the few elements after the last whole vector: lane e of the team takes element e (the
    // lanes behind them re-read the last one), and later stores its code
    float te = 0.0f;
    if (tail) te = Elem<T>::load(s.ptr, r0 + nvec * EPV + min(lane, tail - 1));
    float amax = 0.0f;
#pragma unroll
    for (int k = 0; k < KMAX; k++) amax = fmaxf(amax, vec_absmax<T>(v[k]));
    if (tail) amax = fmaxf(amax, __builtin_fabsf(te));
    amax = team_max<TEAM>(amax, lds);
    const float sc = calc_scale(amax);
    if (lane == 0) {
        if (STAGED) srow[0] = as_u(sc);
        else out[0] = as_u(sc);
    }
    // The elements are unpacked again from the raw vectors: keeping the floats of the
    // maximum search alive until here would double the registers of 16-bit inputs.
#pragma unroll
    for (int k = 0; k < KMAX; k++) asm volatile("" : "+v"(v[k].x), "+v"(v[k].y), "+v"(v[k].z), "+v"(v[k].w));
#pragma unroll
    for (int k = 0; k < KMAX; k++) {
        const int idx = k * TEAM + lane;
        if (idx < nvec) {
            if (STAGED) {
                const u32x2 o = vec_codes<T>(v[k], sc);
                if constexpr (EPV == 4) {
                    srow[1 + idx] = o.x;
                } else {
                    srow[1 + 2 * idx] = o.x;
                    srow[2 + 2 * idx] = o.y;
                }
            } else {
                vec_quant_store<T>(v[k], sc, out + 1, idx);
            }
        }
    }
    // tail codes and the zero pad bytes behind them, one byte per lane (a team has at least 8 lanes)
    if (tail && lane < s.row_bytes - 4 - nvec * EPV) {
        const u32 b = lane < tail ? pack_fp8x4(te * sc, 0.0f, 0.0f, 0.0f) & 0xFFu : 0u;
        const int at = 4 + nvec * EPV + lane;
        if (STAGED) ((LDS_AS uint8_t *)srow)[at] = (uint8_t)b;
        else ((GLOBAL uint8_t *)out)[at] = (uint8_t)b;
    }
}

// Rows of more than 4096 vectors (64 KB; wide kernel only): the first 16
// vectors of a lane stay in registers, up to 15 more are parked in LDS, where
// every lane reads back only what it wrote itself, so rows of up to 7936
// vectors (124 KB) are still read from memory once.  The parked vectors travel
// in three groups of five; the loads of the next group are issued before the
// current one is parked.  What a longer row has beyond 7936 vectors is read
// twice, once for the maximum and once to be quantized.
template <typename T>
DEV void quantize_vec_lds(const Seg &s, const KCall &p, int row, int tid, float *lds, u32x4 *park)
{
    constexpr int KR = 2 * QV, G = TFTQ_Q_PARK_GROUP, NG = TFTQ_Q_PARKED / G;
    static_assert(NG * G == TFTQ_Q_PARKED, "groups of five");
    const bool active = row < s.slice_rows * p.ws;
    GLOBAL u32 *out = as_global<u32>(p.packed + (active ? row_addr(s, p.slot_size, row) : 0));
    if (active && row >= s.m) {
        for (int d = tid; d < (s.row_bytes >> 2); d += TFTQ_WG) out[d] = 0;  // padding row
    }
    if (!active || row >= s.m) return;  // the whole workgroup leaves

    constexpr int EPV = Elem<T>::EPV;
    const int nvec = s.n / EPV;
    const int tail = s.n - nvec * EPV;
    const int64_t r0 = (int64_t)row * s.row_stride;
    GLOBAL const u32x4_a2 *in = as_global<const u32x4_a2>(s.ptr + r0 * Elem<T>::ESZ);
    const int dup = dup_vec_offset(in, nvec);
    u32x4 v[KR], w[2][G];
#pragma unroll
    for (int k = 0; k < KR; k++) v[k] = LOAD_STREAM(vec_or_dup(in, k * TFTQ_WG + tid, nvec, dup));
#pragma unroll
    for (int k = 0; k < G; k++) w[0][k] = LOAD_STREAM(vec_or_dup(in, (KR + k) * TFTQ_WG + tid, nvec, dup));
    float te = 0.0f;  // lane e takes element e behind the last whole vector (see quantize_vec_k)
    if (tail) te = Elem<T>::load(s.ptr, r0 + nvec * EPV + min(tid, tail - 1));
    float amax = 0.0f;
#pragma unroll
    for (int k = 0; k < KR; k++) amax = fmaxf(amax, vec_absmax<T>(v[k]));
    // the groups this row needs (the launch has LDS for the longest row of the list)
    const int ng = tftq_q_park_groups(nvec);
#pragma unroll
    for (int g = 0; g < NG; g++) {
        if (g < ng) {  // same for the whole workgroup
            if (g + 1 < NG && g + 1 < ng) {
#pragma unroll
                for (int k = 0; k < G; k++)
                    w[(g + 1) & 1][k] = LOAD_STREAM(vec_or_dup(in, (KR + (g + 1) * G + k) * TFTQ_WG + tid, nvec, dup));
            }
#pragma unroll
            for (int k = 0; k < G; k++) {
                amax = fmaxf(amax, vec_absmax<T>(w[g & 1][k]));
                park[(g * G + k) * TFTQ_WG + tid] = w[g & 1][k];
            }
        }
    }
    if (tail) amax = fmaxf(amax, __builtin_fabsf(te));
#pragma nounroll
    for (int base = TFTQ_Q_VECS_LDS; base < nvec; base += 4 * TFTQ_WG) {  // first pass over the rest
        u32x4 x[4];
#pragma unroll
        for (int k = 0; k < 4; k++) x[k] = in[min(base + k * TFTQ_WG + tid, nvec - 1)];
#pragma unroll
        for (int k = 0; k < 4; k++) amax = fmaxf(amax, vec_absmax<T>(x[k]));
    }
    amax = team_max<256>(amax, lds);
    const float sc = calc_scale(amax);
    if (tid == 0) out[0] = as_u(sc);
#pragma unroll
    for (int k = 0; k < KR; k++) asm volatile("" : "+v"(v[k].x), "+v"(v[k].y), "+v"(v[k].z), "+v"(v[k].w));
#pragma unroll
    for (int k = 0; k < KR; k++) {
        const int idx = k * TFTQ_WG + tid;
        if (idx < nvec) vec_quant_store<T>(v[k], sc, out + 1, idx);
    }
#pragma unroll
    for (int k = 0; k < TFTQ_Q_PARKED; k++) {
        const int idx = (KR + k) * TFTQ_WG + tid;
        if (idx < nvec) vec_quant_store<T>(park[k * TFTQ_WG + tid], sc, out + 1, idx);
    }
#pragma nounroll
    for (int base = TFTQ_Q_VECS_LDS; base < nvec; base += 4 * TFTQ_WG) {  // second pass over the rest
        u32x4 x[4];
#pragma unroll
        for (int k = 0; k < 4; k++) x[k] = LOAD_STREAM(in + min(base + k * TFTQ_WG + tid, nvec - 1));
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int idx = base + k * TFTQ_WG + tid;
            if (idx < nvec) vec_quant_store<T>(x[k], sc, out + 1, idx);
        }
    }
    if (tail && tid < s.row_bytes - 4 - nvec * EPV) {  // tail codes and the zero pad bytes behind them
        const u32 b = tid < tail ? pack_fp8x4(te * sc, 0.0f, 0.0f, 0.0f) & 0xFFu : 0u;
        ((GLOBAL uint8_t *)out)[4 + nvec * EPV + tid] = (uint8_t)b;
    }
}

template <typename T, int TEAM, bool WIDE>
DEV void quantize_vec(const Seg &s, const KCall &p, int row, int lane, float *lds, u32x4 *park)
{
    // same branch for the whole workgroup
    const int nvec = s.n / Elem<T>::EPV;
    if (nvec <= (QV / 2) * TEAM) quantize_vec_k<T, TEAM, QV / 2>(s, p, row, lane, lds);
    else if (TEAM < 256 || nvec <= TFTQ_Q_VECS) quantize_vec_k<T, TEAM, QV>(s, p, row, lane, lds);
    else if (WIDE && nvec <= TFTQ_Q_VECS_WIDE) quantize_vec_k<T, TEAM, 2 * QV>(s, p, row, lane, lds);
    else if (WIDE) quantize_vec_lds<T>(s, p, row, lane, lds, park);
    // else: the planner launches the wide kernel, with its LDS, for plans that have such rows
}

// The TFTQ_WG / TEAM rows of workgroup blk.  When they are all real rows of one slot (all
// but the workgroups at the end of a slot or of the tensor) and fit the staging buffer,
// their packed rows are assembled in LDS and written as one span; otherwise row by row.
template <typename T, int TEAM, bool WIDE>
DEV void quantize_vec_rows(const Seg &s, const KCall &p, int blk, int tid, float *lds, u32x4 *park, uint8_t *stage)
{
    constexpr int R = TFTQ_WG / TEAM;
    const int r0 = blk * R;
    const int team = TEAM == 64 ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid / TEAM;
    const int lane = tid & (TEAM - 1);
    {
        constexpr int KMAX = WIDE && TEAM == 256 ? 2 * QV : QV;  // vectors per lane that the kernel keeps in registers
        constexpr int STAGE_BYTES = WIDE ? Q_STAGE_BYTES_WIDE : Q_STAGE_BYTES;
        const int nvec = s.n / Elem<T>::EPV;
        const int last = r0 + R - 1;
        if (last < s.m && nvec <= KMAX * TEAM) {
            const int slot = r0 / s.slice_rows;
            const int j = r0 - slot * s.slice_rows;
            uint8_t *g0 = p.packed + (int64_t)slot * p.slot_size + s.slot_off + (int64_t)j * s.row_bytes;
            const int mis = (int)((uintptr_t)g0 & 127u);
            const int len = R * s.row_bytes;
            if (j + R <= s.slice_rows && mis + len <= STAGE_BYTES) {  // same for the whole workgroup
                LDS_AS u32 *srow = (LDS_AS u32 *)(LDS_AS uint8_t *)(stage + mis + team * s.row_bytes);
                if (nvec <= (QV / 2) * TEAM) quantize_vec_k<T, TEAM, QV / 2, true>(s, p, r0 + team, lane, lds, srow);
                else if (KMAX == QV || nvec <= QV * TEAM) quantize_vec_k<T, TEAM, QV, true>(s, p, r0 + team, lane, lds, srow);
                else quantize_vec_k<T, TEAM, KMAX, true>(s, p, r0 + team, lane, lds, srow);
                __syncthreads();
                copy_out_span(stage, g0, len, tid);
                return;
            }
        }
    }
    quantize_vec<T, TEAM, WIDE && TEAM == 256>(s, p, r0 + team, lane, lds, park);
}

// Any strides, any alignment, any n: element loads, two passes over the row
// (the second one is served by the caches).
template <typename T, int TEAM>
DEV void quantize_gen(const Seg &s, const KCall &p, int row, int lane)
{
    const bool active = row < s.slice_rows * p.ws;
    if (!active) return;
    GLOBAL u32 *out = as_global<u32>(p.packed + row_addr(s, p.slot_size, row));
    const int ndw = (s.row_bytes >> 2) - 1;
    if (row >= s.m) {
        for (int d = lane; d <= ndw; d += TEAM) out[d] = 0;
        return;
    }
    const uint64_t base = s.ptr;
    const int64_t r0 = (int64_t)row * s.row_stride;
    float amax = 0.0f;
    for (int c = lane; c < s.n; c += TEAM)
        amax = fmaxf(amax, __builtin_fabsf(Elem<T>::load(base, r0 + (int64_t)c * s.col_stride)));
    amax = team_max<TEAM>(amax, nullptr);
    const float sc = calc_scale(amax);
    if (lane == 0) out[0] = as_u(sc);
    for (int d = lane; d < ndw; d += TEAM) {
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int c = 4 * d + e;
            const float x = c < s.n ? Elem<T>::load(base, r0 + (int64_t)c * s.col_stride) : 0.0f;
            y[e] = x * sc;
        }
        u32 w = pack_fp8x4(y[0], y[1], y[2], y[3]);
        const int tail = s.n - 4 * d;  // codes of this dword that belong to the row
        if (tail < 4) w &= (1u << (8 * tail)) - 1u;  // zero padding, whatever 0 * sc gave
        out[1 + d] = w;
    }
}

// Rows of one column (1-D tensors, quantization.py:487-488): a row is its own
// maximum, so the code is +-448 (or 0) and all information is in the scale.
// [scale, code] of one row
DEV u32x2 quantize_one(float x)
{
    // maximum with 0 as for longer rows: a NaN element is ignored (:131-143)
    const float sc = calc_scale(fmaxf(0.0f, __builtin_fabsf(x)));
    u32x2 o;
    o.x = as_u(sc);
    o.y = pack_fp8x4(x * sc, 0.0f, 0.0f, 0.0f) & 0xFFu;
    return o;
}

// Any element stride: four rows per lane, interleaved so that every 8-byte
// [scale, code] store of a wavefront is contiguous.
template <typename T, int ROWS>
DEV void quantize_col1_strided(const Seg &s, const KCall &p, int row0, int tid)
{
    const int m_pad = s.slice_rows * p.ws;
    const float inv = 1.0f / (float)s.slice_rows;
    float x[ROWS];
#pragma unroll
    for (int k = 0; k < ROWS; k++) {
        const int row = min(row0 + k * TFTQ_WG + tid, s.m - 1);
        x[k] = s.m > 0 ? Elem<T>::load(s.ptr, (int64_t)row * s.row_stride) : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < ROWS; k++) {
        const int row = row0 + k * TFTQ_WG + tid;
        if (row < m_pad) {
            u32x2 o = {0u, 0u};  // padding rows stay zero
            if (row < s.m) o = quantize_one(x[k]);
            *(GLOBAL u32x2_a4 *)as_global<u32>(p.packed + row_addr_fast(s, p.slot_size, row, inv)) = o;
        }
    }
}

// Contiguous elements: a lane takes PAIRS pairs of neighbouring rows, so that it
// reads two elements with one load (a wavefront reads 256 or 512 contiguous
// bytes per load even for 2-byte elements) and writes their two packed rows
// with one 16-byte streaming store (a wavefront writes 1 KB of whole lines).
// A pair that straddles the end of a slot or of the tensor is stored row by row.
template <typename T, int PAIRS>
DEV void quantize_col1(const Seg &s, const KCall &p, int row0, int tid)
{
    constexpr int ROWS = PAIRS > 1 ? 4 : 2;  // of a step of the strided path
    if (s.row_stride != 1) {  // same for the whole workgroup
#pragma nounroll
        for (int r = 0; r < 2 * PAIRS * TFTQ_WG && row0 + r < s.slice_rows * p.ws; r += ROWS * TFTQ_WG)
            quantize_col1_strided<T, ROWS>(s, p, row0 + r, tid);
        return;
    }
    const int m_pad = s.slice_rows * p.ws;
    const float inv = 1.0f / (float)s.slice_rows;
    float x[PAIRS][2];
#pragma unroll
    for (int k = 0; k < PAIRS; k++) {
        const int row = row0 + 2 * (k * TFTQ_WG + tid);
        x[k][0] = x[k][1] = 0.0f;
        if (row + 1 < s.m) Elem<T>::load2(s.ptr, row, x[k][0], x[k][1]);
        else if (row < s.m) x[k][0] = Elem<T>::load(s.ptr, row);
    }
#pragma unroll
    for (int k = 0; k < PAIRS; k++) {
        const int row = row0 + 2 * (k * TFTQ_WG + tid);
        if (row >= m_pad) continue;
        u32x2 a = {0u, 0u}, b = {0u, 0u};  // padding rows stay zero
        if (row < s.m) a = quantize_one(x[k][0]);
        if (row + 1 < s.m) b = quantize_one(x[k][1]);
        int slot = (int)((float)row * inv);  // off by at most one
        int j = row - slot * s.slice_rows;
        if (j < 0) { --slot; j += s.slice_rows; }
        if (j >= s.slice_rows) { ++slot; j -= s.slice_rows; }
        GLOBAL u32 *dst = as_global<u32>(p.packed + (int64_t)slot * p.slot_size + s.slot_off + (int64_t)j * 8);
        if (j + 1 < s.slice_rows) {  // the next row follows in the same slot (and row + 1 < m_pad)
            const u32x4 o = {a.x, a.y, b.x, b.y};
            STORE_STREAM(o, (GLOBAL u32x4_a4 *)dst);
        } else {
            *(GLOBAL u32x2_a4 *)dst = a;
            if (row + 1 < m_pad)
                *(GLOBAL u32x2_a4 *)as_global<u32>(p.packed + row_addr_fast(s, p.slot_size, row + 1, inv)) = b;
        }
    }
}

// Short contiguous rows of 1 to 32 16-byte vectors (K_VECS, shape in tftq_device.h).  A row
// whose length is not a whole number of vectors has its last vector moved back so that it
// ends with the row: it overlaps its neighbour, whose elements count twice for the maximum
// (no matter) and whose codes are written twice with the same values.
// First column of vector idx of a row of n columns.
template <typename T>
DEV int small_vec_col(int idx, int n)
{
    return min(idx * Elem<T>::EPV, n - Elem<T>::EPV);
}

DEV void put8(LDS_AS uint8_t *q, u32 v) { *q = (uint8_t)v; }
DEV void put8(GLOBAL uint8_t *q, u32 v) { *q = (uint8_t)v; }
DEV void put32(LDS_AS uint8_t *q, u32 v) { *(LDS_AS u32 *)q = v; }
DEV void put32(GLOBAL uint8_t *q, u32 v) { *(GLOBAL u32 *)q = v; }
DEV void put64(LDS_AS uint8_t *q, u32x2 v) { *(LDS_AS u32x2_a4 *)q = v; }
DEV void put64(GLOBAL uint8_t *q, u32x2 v) { *(GLOBAL u32x2_a4 *)q = v; }

// The codes o of vector idx (of nv) into the packed row at `row` (LDS or global memory); the
// lane of the last vector also clears the pad bytes behind the row's last code.
// TAIL false: rows of whole vectors, which have neither a moved vector nor pad bytes.
template <typename T, bool TAIL, typename P>
DEV void put_small_codes(P row, int idx, int nv, int n, int row_bytes, const u32x2 o)
{
    constexpr int EPV = Elem<T>::EPV;
    if constexpr (!TAIL) {
        if constexpr (EPV == 4) put32(row + 4 + idx * EPV, o.x);
        else put64(row + 4 + idx * EPV, o);
        return;
    }
    const int col = small_vec_col<T>(idx, n);
    if ((col & 3) == 0) {
        if constexpr (EPV == 4) put32(row + 4 + col, o.x);
        else put64(row + 4 + col, o);
    } else {  // the moved last vector of a row that is not a whole number of dwords
#pragma unroll
        for (int e = 0; e < EPV; e++) put8(row + 4 + col + e, (e < 4 ? o.x : o.y) >> (8 * (e & 3)));
    }
    if (idx == nv - 1)
        for (int b = 4 + n; b < row_bytes; b++) put8(row + b, 0u);
}

// Scale of the row whose vectors a lane holds in v (maximum over the lanes of its team).
template <typename T, int C>
DEV float small_row_scale(const u32x4 (&v)[C], const SmallShape &h)
{
    float a = 0.0f;
#pragma unroll
    for (int k = 0; k < C; k++) {
        a = fmaxf(a, vec_absmax<T>(v[k]));
    }
    if (h.lt >= 1) a = fmaxf(a, dpp_mov<0xB1>(a));   // quad_perm [1,0,3,2]
    if (h.lt >= 2) a = fmaxf(a, dpp_mov<0x4E>(a));   // quad_perm [2,3,0,1]
    if (h.lt >= 3) a = fmaxf(a, dpp_mov<0x141>(a));  // row_half_mirror
    if (h.lt >= 4) a = fmaxf(a, dpp_mov<0x140>(a));  // row_mirror: all 16 lanes of a row agree
    if (h.lt >= 5) {  // same for the whole workgroup
        const float lo = fmaxf(bcast_lane(a, 0), bcast_lane(a, 16)), hi = fmaxf(bcast_lane(a, 32), bcast_lane(a, 48));
        a = (threadIdx.x & 32) ? hi : lo;
    }
    return calc_scale(a);
}

// Rows RBEG * teams .. REND * teams - 1 of the workgroup's rows (those up to `last`)
// through the LDS stage: g0 is the address of the workgroup's first packed row.
template <typename T, int C, bool TAIL, int ROWS, int RBEG, int REND>
DEV void quantize_small_span(const Seg &s, const SmallShape &h, const u32x4 (&v)[ROWS][C], int row0, int last,
                             uint8_t *g0, uint8_t *stage, int tid)
{
    const int nvec = tftq_small_nvec(s.n, Elem<T>::ESZ);
    const int first = row0 + RBEG * h.teams;
    if (first > last) return;  // same for the whole workgroup
    uint8_t *gp = g0 + (int64_t)(RBEG * h.teams) * s.row_bytes;
    const int mis = (int)((uintptr_t)gp & 127u);
    const int len = (min(last, row0 + REND * h.teams - 1) - first + 1) * s.row_bytes;
#pragma unroll
    for (int r = RBEG; r < REND; r++) {
        const int row = row0 + r * h.teams + h.t;
        const float sc = small_row_scale<T, C>(v[r], h);
        if (row > last) continue;
        LDS_AS uint8_t *srow = (LDS_AS uint8_t *)(stage + mis + ((r - RBEG) * h.teams + h.t) * s.row_bytes);
        if (row >= s.m) {  // padding row: zero (:93-95 on a zero-filled buffer)
            for (int d = h.l; d < (s.row_bytes >> 2); d += h.team) ((LDS_AS u32 *)srow)[d] = 0;
            continue;
        }
        if (h.l == 0) *(LDS_AS u32 *)srow = as_u(sc);
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int idx = k * h.team + h.l;
            if (idx >= nvec) continue;
            const u32x4 x = v[r][k];
            put_small_codes<T, TAIL>(srow, idx, nvec, s.n, s.row_bytes, vec_codes<T>(x, sc));
        }
    }
    __syncthreads();
    copy_out_span(stage, gp, len, tid);
}

// The rows of a workgroup are neighbours; when they lie in one slot their packed rows are
// one span of bytes, which goes through LDS (copy_out_span) in two halves (rows of 8 to 64
// 16-bit columns make up to 24 KB per workgroup, more than the stage holds).
// VECS: vectors per lane, 8 (K_VECS) or 2 (K_VECS_FEW).
template <typename T, int C, bool TAIL, int VECS>
DEV void quantize_small_c(const Seg &s, const KCall &p, int blk, int tid, const SmallShape &h, uint8_t *stage)
{
    constexpr int ROWS = VECS / C;  // C vectors per lane and row, ROWS rows per lane
    const int nvec = tftq_small_nvec(s.n, Elem<T>::ESZ);
    const int nrows = h.teams * ROWS;
    const int row0 = blk * nrows;
    const int m_pad = s.slice_rows * p.ws;
    const float inv = 1.0f / (float)s.slice_rows;

    u32x4 v[ROWS][C];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const int row = row0 + r * h.teams + h.t;
        const int64_t e0 = (int64_t)min(row, s.m - 1) * s.row_stride;  // s.m >= 1: there are rows
        // a lane past the row's last vector re-reads that one: a duplicate cannot change the maximum
        if constexpr (TAIL) {
#pragma unroll
            for (int k = 0; k < C; k++) {
                const int col = small_vec_col<T>(min(k * h.team + h.l, nvec - 1), s.n);
                v[r][k] = LOAD_STREAM(as_global<const u32x4_a2>(s.ptr + (e0 + col) * Elem<T>::ESZ));
            }
        } else {
            GLOBAL const u32x4_a2 *in = as_global<const u32x4_a2>(s.ptr + e0 * Elem<T>::ESZ);
#pragma unroll
            for (int k = 0; k < C; k++) v[r][k] = LOAD_STREAM(in + min(k * h.team + h.l, nvec - 1));
        }
    }
    {
        // the workgroup's rows that exist, row0 .. last, and the slot of the first one
        const int last = min(row0 + nrows, m_pad) - 1;
        int slot0 = (int)((float)row0 * inv);
        int j0 = row0 - slot0 * s.slice_rows;
        if (j0 < 0) { --slot0; j0 += s.slice_rows; }
        if (j0 >= s.slice_rows) { ++slot0; j0 -= s.slice_rows; }
        if (j0 + (last - row0) < s.slice_rows) {  // one slot: one span.  Same for the whole workgroup
            // the marker keeps the compiler from moving what this path and the one below have in
            // common, the scales of all rows, in front of the branch (20 more registers)
            asm volatile("; rows through the stage");
            uint8_t *g0 = p.packed + (int64_t)slot0 * p.slot_size + s.slot_off + (int64_t)j0 * s.row_bytes;
            if constexpr (VECS == TFTQ_SMALL_VECS) {
                quantize_small_span<T, C, TAIL, ROWS, 0, ROWS / 2>(s, h, v, row0, last, g0, stage, tid);
                __syncthreads();  // the first half has been copied out of the stage
                quantize_small_span<T, C, TAIL, ROWS, ROWS / 2, ROWS>(s, h, v, row0, last, g0, stage, tid);
            } else {
                quantize_small_span<T, C, TAIL, ROWS, 0, ROWS>(s, h, v, row0, last, g0, stage, tid);
            }
            return;
        }
    }
    asm volatile("; rows straight from the registers");
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const int row = row0 + r * h.teams + h.t;
        const float sc = small_row_scale<T, C>(v[r], h);
        if (row >= m_pad) continue;
        GLOBAL uint8_t *out = as_global<uint8_t>(p.packed + row_addr_fast(s, p.slot_size, row, inv));
        if (row >= s.m) {
            // padding row: the reference leaves it zero (:93-95 on a zero-filled buffer)
            for (int d = h.l; d < (s.row_bytes >> 2); d += h.team) ((GLOBAL u32 *)out)[d] = 0;
            continue;
        }
        if (h.l == 0) *(GLOBAL u32 *)out = as_u(sc);
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int idx = k * h.team + h.l;
            if (idx >= nvec) continue;
            const u32x4 x = v[r][k];
            put_small_codes<T, TAIL>(out, idx, nvec, s.n, s.row_bytes, vec_codes<T>(x, sc));
        }
    }
}

template <typename T, int VECS>
DEV void quantize_small(const Seg &s, const KCall &p, int blk, int tid, uint8_t *stage)
{
    const SmallShape h = small_shape(tftq_small_nvec(s.n, Elem<T>::ESZ), tid, ST_Q);
    // one or two vectors per lane (tftq_small_shape); same branch for the whole workgroup
    if (s.n % Elem<T>::EPV) {
        if (h.c == 1) quantize_small_c<T, 1, true, VECS>(s, p, blk, tid, h, stage);
        else quantize_small_c<T, 2, true, VECS>(s, p, blk, tid, h, stage);
    } else if (h.c == 1) quantize_small_c<T, 1, false, VECS>(s, p, blk, tid, h, stage);
    else quantize_small_c<T, 2, false, VECS>(s, p, blk, tid, h, stage);
}

template <typename T, bool WIDE, typename A>
DEV void quantize_workgroup(const A &args)
{
    constexpr bool FEW = !WIDE;  // the kinds for little work (pick_few_kinds)
    __shared__ float lds[4];
    __shared__ __align__(16) uint8_t stage_regular[WIDE ? 16 : Q_STAGE_BYTES];  // see copy_out_span
    // Dynamic LDS of the wide kernel: Q_STAGE_BYTES_WIDE as its stage, or the 40 or 60 KB that the
    // longest row of the plan parks there (which limits a CU to three or two workgroups); a
    // workgroup uses it for one or the other.
    extern __shared__ u32x4 park[];
    uint8_t *stage = WIDE ? (uint8_t *)park : stage_regular;
    Seg s;
    KCall p;
    int blk;
    if (!locate<ST_Q>(args, p, s, blk)) return;
    const int tid = threadIdx.x;
    switch (s.kind[ST_Q]) {
    case K_VEC256: quantize_vec_rows<T, 256, WIDE>(s, p, blk, tid, lds, park, stage); break;
    case K_VEC64: quantize_vec_rows<T, 64, WIDE>(s, p, blk, tid, lds, park, stage); break;
    case K_VEC32: quantize_vec_rows<T, 32, WIDE>(s, p, blk, tid, lds, park, stage); break;
    case K_VEC16: quantize_vec_rows<T, 16, WIDE>(s, p, blk, tid, lds, park, stage); break;
    case K_VEC8: quantize_vec_rows<T, 8, WIDE>(s, p, blk, tid, lds, park, stage); break;
    case K_GEN64:
        quantize_gen<T, 64>(s, p, blk * 4 + __builtin_amdgcn_readfirstlane(tid >> 6), tid & 63);
        break;
    case K_GEN8: quantize_gen<T, 8>(s, p, blk * 32 + (tid >> 3), tid & 7); break;
    case K_GEN1: quantize_gen<T, 1>(s, p, blk * 256 + tid, 0); break;
    case K_COL1: quantize_col1<T, TFTQ_COL1_PAIRS_Q>(s, p, blk * tftq_col1_rows_per_wg(ST_Q), tid); break;
    case K_VECS: quantize_small<T, TFTQ_SMALL_VECS>(s, p, blk, tid, stage); break;
    case K_COL1_FEW:
        if constexpr (FEW) quantize_col1<T, 1>(s, p, blk * tftq_col1_rows_per_wg(ST_Q, true), tid);
        break;
    case K_VECS_FEW:
        if constexpr (FEW) quantize_small<T, TFTQ_SMALL_VECS_FEW>(s, p, blk, tid, stage);
        break;
    default: break;
    }
}

// The wide variant is held to 128 registers (four waves per SIMD instead of three at the 153 to
// 166 it would take): lists that mix rows of more than 32 KB with shorter ones run whole in
// it, and the shorter rows gain 10 % (a Llama-3-70B layer bucket: 464 -> 420 us).
template <typename T, typename A, bool WIDE>
__global__ __launch_bounds__(TFTQ_WG, WIDE ? 4 : 1) void k_quantize(const A args)
{
    quantize_workgroup<T, WIDE>(args);
}
template <typename T, bool WIDE>
__global__ __launch_bounds__(TFTQ_WG, WIDE ? 4 : 1) void k_quantize_one(TFTQ_ONE_PARAMS)
{
    quantize_workgroup<T, WIDE>(one_of(TFTQ_ONE));
}

// ---------------------------------------------------------------------------
// quantize, tensors whose columns are contiguous in memory (K_COLS)
// ---------------------------------------------------------------------------
// A transposed matrix: a row's elements are a whole column length apart, a column's lie side by
// side.  A lane takes 16 bytes of a column, 8 (fp32: 4) rows, of four neighbouring columns: it then
// holds one dword of codes of each of these rows, with no exchange between lanes.  Only the row
// maxima go through LDS, and the packed rows where a block's fit (they are one span of bytes:
// copy_out_span).  A block of G such groups of rows stays in the registers of a workgroup of 512
// lanes, up to NS steps of 2048 / G columns, so that the tensor is read once; what a row has beyond
// that is read twice (in 2 groups; more groups hold their rows whole).  Bound by memory where 8 or more groups make whole lines of
// what a block reads; with 2 groups it uses 32 bytes of a line and the L1's requests in flight are the
// limit.  bf16, 8 slots, 2 groups and dwords stored from the registers -> with the groups that
// pick_groups takes and the stage: [285326, 147] 101 -> 26 us (4.8 TB/s), [1310720, 32] 447 -> 29, [41943, 1000]
// 50 -> 22, [20971, 2000] 46 -> 23, [6990, 6000] 48 -> 34; fp32 [285326, 147] 161 -> 42, [41943, 1000] 75 -> 46.
// [4096, 14336] in 2 groups, 66 to 69 us: with blocks of 32 rows 101 (half the compute units idle), workgroups of
// 256 lanes 89 (half of the row read twice), of 1024 lanes 72, streaming loads 77 (neighbouring blocks
// share lines); a launch for the maxima and one for tiles of 64 rows 82 us.  Where the blocks lose against
// teams of lanes (few rows per slot) the planner leaves them out: pick_column_kinds.
// REST: with the first pass over what a row has beyond NS steps, whether a row has that or not.  It changes the
// order of the other loads: with it the compiler computes maxima between them, with some 8 in flight, without
// it all loads of up to 8 steps come first.  The former suits blocks that have a compute unit's L1 to
// themselves for long enough, the latter a machine full of them (see k_quantize_cols_two).
template <typename T, int G, int NS, int STAGE, bool REST = true>
DEV void quantize_cols(const Seg &s, const KCall &p, int blk, int tid, uint8_t *stage, float *scale)
{
    constexpr int EPV = Elem<T>::EPV, ESZ = Elem<T>::ESZ, K = 64 / G, RB = G * EPV;
    constexpr int WAVES = TFTQ_QC_WG / 64, STEP = 4 * K * WAVES;  // columns per step
    constexpr int RPD = 4 / ESZ;                                  // rows per dword of a column
    constexpr int SETS = G <= 16 ? 4 : 2;                         // of lanes that hold all groups, per wavefront
    constexpr bool STAGED = RB * (4 + NS * STEP) + 127 <= STAGE;  // the block's packed rows fit the stage
    static_assert(SETS * WAVES * RB * 4 <= STAGE, "the maxima fit the stage");
    float *part = (float *)stage;
    const int per_slot = (s.slice_rows + RB - 1) / RB;
    const int slot = blk / per_slot;
    const int j0 = (blk - slot * per_slot) * RB;
    const int srow = slot * s.slice_rows;  // the slot's first row
    const int real = min(max(s.m - srow, 0), s.slice_rows);
    GLOBAL uint8_t *g0 = as_global<uint8_t>(p.packed + (int64_t)slot * p.slot_size + s.slot_off + (int64_t)j0 * s.row_bytes);
    if (!STAGED || j0 >= real) {   // padding rows: zero (:93-95 on a zero-filled buffer)
        const int z0 = max(real - j0, 0), z1 = min(RB, s.slice_rows - j0);
        for (int z = z0; z < z1; z++)
            for (int d = tid; d < (s.row_bytes >> 2); d += TFTQ_QC_WG) ((GLOBAL u32 *)(g0 + (int64_t)z * s.row_bytes))[d] = 0;
    }
    if (j0 >= real) return;  // the whole workgroup
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int g = l & (G - 1), k = l / G;
    const int ndw = (s.row_bytes >> 2) - 1;
    // the lane's rows; the last group of the tensor is moved back to end with it (its rows are
    // another lane's too: both write the same bytes)
    const int first = min(srow + j0 + g * EPV, s.m - EPV);
    const int jf = first - srow - j0, jstop = min(RB, real - j0);  // rows jf + i in [0, jstop) are written
    const uint64_t col0 = s.ptr + (uint64_t)((int64_t)first * ESZ);
    const int64_t cs = s.col_stride * ESZ;
    const int c0 = 4 * (wave * K + k);
    auto load = [&](u32x4 (&v)[4], int base) {
#pragma unroll
        for (int e = 0; e < 4; e++)  // columns past the last one re-read it
            v[e] = *as_global<const u32x4_a2>(col0 + (uint64_t)((int64_t)min(base + c0 + e, s.n - 1) * cs));
    };
    float amax[EPV];
#pragma unroll
    for (int i = 0; i < EPV; i++) amax[i] = 0.0f;
    auto maxima = [&](const u32x4 (&v)[4]) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float f[EPV];
            Elem<T>::unpack(v[e], f);
#pragma unroll
            for (int i = 0; i < EPV; i++) amax[i] = fmaxf(amax[i], __builtin_fabsf(f[i]));
        }
    };
    u32x4 v[NS][4];
#pragma unroll
    for (int t = 0; t < NS; t++) load(v[t], t * STEP);
#pragma unroll
    for (int t = 0; t < NS; t++) maxima(v[t]);
    if constexpr (REST) {
#pragma nounroll
        for (int base = NS * STEP; base < s.n; base += STEP) {  // first pass over the rest
            u32x4 x[4];
            load(x, base);
            maxima(x);
        }
    }
#pragma unroll
    for (int i = 0; i < EPV; i++) {  // over the lanes of the same group in a row of 16
        if constexpr (G <= 8) amax[i] = fmaxf(amax[i], dpp_mov<0x128>(amax[i]));  // row_ror:8
        if constexpr (G <= 4) amax[i] = fmaxf(amax[i], dpp_mov<0x124>(amax[i]));  // row_ror:4
        if constexpr (G <= 2) amax[i] = fmaxf(amax[i], dpp_mov<0x122>(amax[i]));  // row_ror:2
        if ((l & 15) < G) part[(wave * SETS + l / (64 / SETS)) * RB + g * EPV + i] = amax[i];
    }
    static_assert(G == 2 || G == 4 || G == 8 || G == 16 || G == 32, "the rotations above");
    __syncthreads();
    if (tid < RB) {
        float a = 0.0f;
#pragma unroll
        for (int w = 0; w < SETS * WAVES; w++) a = fmaxf(a, part[w * RB + tid]);
        const float sc = calc_scale(a);
        scale[tid] = sc;
        if constexpr (!STAGED) {
            const int j = min(srow + j0 + tid / EPV * EPV, s.m - EPV) - srow - j0 + tid % EPV;
            if (j >= 0 && j < jstop) *(GLOBAL u32 *)(g0 + (int64_t)j * s.row_bytes) = as_u(sc);
        }
    }
    __syncthreads();  // the maxima have been read: the stage is free
    LDS_AS uint8_t *span = (LDS_AS uint8_t *)(stage + (int)((uintptr_t)g0 & 127u));  // STAGED: where g0 is
    if constexpr (STAGED) {
        const int j = min(srow + j0 + tid / EPV * EPV, s.m - EPV) - srow - j0 + tid % EPV;
        if (tid < RB && j >= 0 && j < jstop) *(LDS_AS u32 *)(span + j * s.row_bytes) = as_u(scale[tid]);
        for (int z = real - j0; z < min(RB, s.slice_rows - j0); z++)  // padding rows
            for (int d = tid; d < (s.row_bytes >> 2); d += TFTQ_QC_WG) ((LDS_AS u32 *)(span + z * s.row_bytes))[d] = 0;
    }
    float sc[EPV];
#pragma unroll
    for (int i = 0; i < EPV; i++) sc[i] = scale[g * EPV + i];
    GLOBAL uint8_t *out = g0 + (int64_t)jf * s.row_bytes + 4;
    auto store = [&](const u32x4 (&v)[4], int base) {
        const int d = (base + c0) >> 2;  // the lane's dword of the payload
        if (d >= ndw) return;
        const int over = 4 * d + 4 - s.n;  // columns of the dword past the last one
        const u32 mask = over > 0 ? 0xFFFFFFFFu >> (8 * over) : 0xFFFFFFFFu;
#pragma unroll
        for (int w = 0; w < 4; w++) {  // dword w of the four vectors: rows RPD * w ...
            float f[4][RPD];
#pragma unroll
            for (int e = 0; e < 4; e++) unpack_dword<T>(v[e][w], f[e]);
#pragma unroll
            for (int h = 0; h < RPD; h++) {
                const int i = RPD * w + h;
                const u32 o = pack_fp8x4(f[0][h] * sc[i], f[1][h] * sc[i], f[2][h] * sc[i], f[3][h] * sc[i]) & mask;
                if (jf + i >= 0 && jf + i < jstop) {
                    if constexpr (STAGED) ((LDS_AS u32 *)(span + (jf + i) * s.row_bytes + 4))[d] = o;
                    // plain stores: a packed row starts anywhere in its line, the L2 puts the runs together
                    else ((GLOBAL u32 *)(out + (int64_t)i * s.row_bytes))[d] = o;
                }
            }
        }
    };
#pragma unroll
    for (int t = 0; t < NS; t++) {
#pragma unroll
        for (int e = 0; e < 4; e++) asm volatile("" : "+v"(v[t][e].x), "+v"(v[t][e].y), "+v"(v[t][e].z), "+v"(v[t][e].w));
    }
#pragma unroll
    for (int t = 0; t < NS; t++) store(v[t], t * STEP);
#pragma nounroll
    for (int base = NS * STEP; base < s.n; base += STEP) {  // second pass over the rest
        u32x4 x[4];
        load(x, base);
        store(x, base);
    }
    if constexpr (STAGED) {
        __syncthreads();
        copy_out_span<TFTQ_QC_WG>(stage, (uint8_t *)g0, min(RB, s.slice_rows - j0) * s.row_bytes, tid);
    }
}

// Steps that stay in registers: 12 for lists with rows of more than 4 steps (250 registers, two
// wavefronts per SIMD; 14 spill), else 4 (115 registers, four).
constexpr int QC_MOST = 12;
// The stage: all packed rows of a block of up to 4 steps, in fp32 also those of 12 steps of 4 groups.  2 groups do
// without in fp32 ([41943, 1000] 75 us straight from the registers and 77 through the stage) and beside rows of more
// than 4 steps (bf16 [4096, 8192], [8192, 4096] and [4096, 1024] in one list, 4 slots, 73.6 us through the stage and 70.3).
template <typename T, int NSMAX>
struct ColsStage {
    static constexpr int VECTORS = Elem<T>::ESZ == 4 ? NSMAX : 4;
    static constexpr int BYTES = TFTQ_QC_WG * 4 * VECTORS * Elem<T>::EPV + 32 * Elem<T>::EPV * 4 + 128;
};
constexpr int QC_LEAST_STAGE = 4096;  // for the maxima of up to 4 groups alone
// The variants that tftq_qc_has names.
template <typename T, int G, int NSMAX>
DEV void quantize_cols_steps(const Seg &s, const KCall &p, int blk, int tid, uint8_t *stage, float *scale)
{
    constexpr int STAGE = ColsStage<T, NSMAX>::BYTES, LG = __builtin_ctz(G);
    constexpr bool DIRECT = G == 2 && (Elem<T>::ESZ == 4 || NSMAX > 4);
    const int steps = tftq_qc_steps(s.n, LG);  // same for the whole workgroup
    constexpr int SHORT = DIRECT ? QC_LEAST_STAGE : STAGE;
    if (!tftq_qc_has(LG, 2) || steps <= 1) quantize_cols<T, G, 1, SHORT>(s, p, blk, tid, stage, scale);
    else if constexpr (tftq_qc_has(LG, 2)) {
        if (steps <= 2) quantize_cols<T, G, 2, SHORT>(s, p, blk, tid, stage, scale);
        else if (NSMAX == 4 || !tftq_qc_has(LG, 12) || steps <= 4) quantize_cols<T, G, 4, SHORT>(s, p, blk, tid, stage, scale);
        else if constexpr (NSMAX > 4 && tftq_qc_has(LG, 12)) {
            constexpr bool EIGHT = tftq_qc_has(LG, 8);
            if (EIGHT && steps <= 8) quantize_cols<T, G, EIGHT ? 8 : NSMAX, SHORT>(s, p, blk, tid, stage, scale);
            else quantize_cols<T, G, NSMAX, Elem<T>::ESZ == 4 && G == 4 ? STAGE : QC_LEAST_STAGE>(s, p, blk, tid, stage, scale);
        }
    }
}
template <typename T, int NSMAX, typename A>
DEV void quantize_cols_workgroup(const A &args)
{
    __shared__ __align__(16) uint8_t stage[ColsStage<T, NSMAX>::BYTES];  // the rows' maxima, then see copy_out_span
    __shared__ float scale[32 * Elem<T>::EPV];
    Seg s;
    KCall p;
    int blk;
    if (!locate<ST_Q>(args, p, s, blk)) return;
    const int tid = threadIdx.x;
    switch (s.lg_groups) {
    case 5: quantize_cols_steps<T, 32, 4>(s, p, blk, tid, stage, scale); break;
    case 4: quantize_cols_steps<T, 16, 4>(s, p, blk, tid, stage, scale); break;
    case 3: quantize_cols_steps<T, 8, 4>(s, p, blk, tid, stage, scale); break;
    case 2: quantize_cols_steps<T, 4, NSMAX>(s, p, blk, tid, stage, scale); break;
    default: quantize_cols_steps<T, 2, NSMAX>(s, p, blk, tid, stage, scale); break;
    }
}
template <typename T, typename A, int NSMAX>
__global__ __launch_bounds__(TFTQ_QC_WG, NSMAX > 4 ? 2 : 4) void k_quantize_cols(const A args)
{
    quantize_cols_workgroup<T, NSMAX>(args);
}
template <typename T, int NSMAX>
__global__ __launch_bounds__(TFTQ_QC_WG, NSMAX > 4 ? 2 : 4) void k_quantize_cols_one(TFTQ_ONE_PARAMS)
{
    quantize_cols_workgroup<T, NSMAX>(one_of(TFTQ_ONE));
}

// Lists whose tensors all have 2 groups, rows of up to MOST steps: the same straight from the registers, in
// kernels that hold nothing else and leave a compute unit its LDS.  us with the rest's first pass in rows of up to 8 steps / without
// it (kernels of up to 12 steps, 8 slots):
//   bf16 16 blocks of 4500 / 7001 columns 8.1, 9.8 / 9.1, 10.9; 24 of 7500 16.5 / 17.1; 48 18.1 / 18.3; 64 20.0 / 19.7;
//     512 of 8192 76.6 / 70.7; and in the same kernel rows of 9 to 14 steps, [8192, 9000] 88.5 / 77.1, [4096, 14336]
//     67.0 / 62.6, alone, and 70.5 / 68.2 beside [4096, 4096], whose loads the compiler orders differently too;
//   fp32 [1024, 4500] 12.4 / 10.8, [3200, 8000] 47.8 / 40.5, [4999, 8191] 76.9 / 62.6.
// Few blocks in 16 bits, rows of up to 8 steps: with it; and those of up to 4 steps, in a kernel of two workgroups
// per compute unit, which is done sooner than the one with the stage: us with / without the stage [256, 1000] 4.3 /
// 3.7, [2048, 4096] (128 blocks) 12.4 / 11.5, [3072, 3300] 12.5 / 11.9, 256 blocks of 1000, 2000 and 4096 columns
// 5.2, 8.7, 13.3 / 4.8, 8.7, 13.8, 400 of 2000 11.4 / 12.2.
template <typename T, int MOST, typename A>
DEV void quantize_cols_two(const A &args)
{
    constexpr bool FEW = MOST < QC_MOST;
    constexpr int STAGE = 4 * TFTQ_QC_WG / 64 * 2 * Elem<T>::EPV * 4;  // for the maxima alone
    __shared__ __align__(16) uint8_t stage[STAGE];
    __shared__ float scale[2 * Elem<T>::EPV];
    Seg s;
    KCall p;
    int blk;
    if (!locate<ST_Q>(args, p, s, blk)) return;
    const int tid = threadIdx.x;
    const int steps = tftq_qc_steps(s.n, 1);  // same for the whole workgroup
    if (steps <= 1) quantize_cols<T, 2, 1, STAGE, FEW>(s, p, blk, tid, stage, scale);
    else if (steps <= 2) quantize_cols<T, 2, 2, STAGE, FEW>(s, p, blk, tid, stage, scale);
    else if (MOST == 4 || steps <= 4) quantize_cols<T, 2, 4, STAGE, FEW>(s, p, blk, tid, stage, scale);
    else if constexpr (MOST > 4) {
        if (MOST == 8 || steps <= 8) quantize_cols<T, 2, 8, STAGE, FEW>(s, p, blk, tid, stage, scale);
        else quantize_cols<T, 2, MOST, STAGE>(s, p, blk, tid, stage, scale);
    }
}
template <typename T, typename A, int MOST>
__global__ __launch_bounds__(TFTQ_QC_WG, MOST > 4 ? 2 : 4) void k_quantize_cols_two(const A args)
{
    quantize_cols_two<T, MOST>(args);
}
template <typename T, int MOST>
__global__ __launch_bounds__(TFTQ_QC_WG, MOST > 4 ? 2 : 4) void k_quantize_cols_two_one(TFTQ_ONE_PARAMS)
{
    quantize_cols_two<T, MOST>(one_of(TFTQ_ONE));
}

template <typename T>
static int launch_qc(const tftq_plan *plan, const KArgs &ka, hipStream_t st)
{
    return with_args(ka, [&](const auto &args) {
        typedef typename std::decay<decltype(args)>::type A;
        constexpr int FEW8 = Elem<T>::ESZ == 2 ? 8 : QC_MOST, FEW4 = Elem<T>::ESZ == 2 ? 4 : QC_MOST;  // (16 bits only)
        if constexpr (std::is_same<A, KOne>::value) {
            auto kernel = k_quantize_cols_one<T, 4>;
            switch (tftq_qc_kernel(*plan)) {
            case QC_ANY_4: break;
            case QC_ANY_12: kernel = k_quantize_cols_one<T, QC_MOST>; break;
            case QC_TWO_4: kernel = k_quantize_cols_two_one<T, FEW4>; break;
            case QC_TWO_8: kernel = k_quantize_cols_two_one<T, FEW8>; break;
            case QC_TWO_12: kernel = k_quantize_cols_two_one<T, QC_MOST>; break;
            }
            return launch_kernel(kernel, ka, args, 0, st, TFTQ_QC_WG);
        } else {
            auto kernel = k_quantize_cols<T, A, 4>;
            switch (tftq_qc_kernel(*plan)) {
            case QC_ANY_4: break;
            case QC_ANY_12: kernel = k_quantize_cols<T, A, QC_MOST>; break;
            case QC_TWO_4: kernel = k_quantize_cols_two<T, A, FEW4>; break;
            case QC_TWO_8: kernel = k_quantize_cols_two<T, A, FEW8>; break;
            case QC_TWO_12: kernel = k_quantize_cols_two<T, A, QC_MOST>; break;
            }
            return launch_kernel(kernel, ka, args, 0, st, TFTQ_QC_WG);
        }
    });
}

template <typename T>
static int launch_q(const tftq_plan *plan, const KArgs &ka, hipStream_t st)
{
    // the parking area also serves as the stage
    const bool wide = plan->wide[ST_Q];
    const unsigned lds = !wide ? 0 : std::max((unsigned)plan->parked * TFTQ_Q_PARK_GROUP * TFTQ_WG * 16u, (unsigned)Q_STAGE_BYTES_WIDE);
    return with_args(ka, [&](const auto &args) {
        typedef typename std::decay<decltype(args)>::type A;
        if constexpr (std::is_same<A, KOne>::value)
            return launch_kernel(wide ? k_quantize_one<T, true> : k_quantize_one<T, false>, ka, args, lds, st);
        else
            return launch_kernel(wide ? k_quantize<T, A, true> : k_quantize<T, A, false>, ka, args, lds, st);
    });
}

extern "C" int tftq_quantize(const tftq_plan *plan, const void *const *tensors, const void *table,
                             void *pointers, void *packed, int64_t packed_bytes, int device, void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    DeviceScope scope(device);
    if (scope.err != hipSuccess) return (int)scope.err;
    if (!plan) return TFTQ_E_ARG;
    const bool rows = plan->nwg[ST_Q] != 0, cols = plan->nwg[ST_QC] != 0;
    int rc = check_call(plan, cols && !rows ? ST_QC : ST_Q, tensors, table, pointers, packed, packed_bytes);
    if (rc || (!rows && !cols)) return rc;
    rc = put_addresses(plan, tensors, pointers, st);
    if (rc) return rc;
    KArgs ka;
    if (rows) {
        fill_args(plan, ST_Q, tensors, table, pointers, packed, PLAIN_CALL, &ka);
        switch (plan->dtype) {
        case TFTQ_F32: rc = launch_q<float>(plan, ka, st); break;
        case TFTQ_F16: rc = launch_q<f16_tag>(plan, ka, st); break;
        case TFTQ_BF16: rc = launch_q<bf16_tag>(plan, ka, st); break;
        default: return TFTQ_E_DTYPE;
        }
        if (rc) return rc;
    }
    if (!cols) return 0;
    fill_args(plan, ST_QC, tensors, table, pointers, packed, PLAIN_CALL, &ka);
    switch (plan->dtype) {
    case TFTQ_F32: return launch_qc<float>(plan, ka, st);
    case TFTQ_F16: return launch_qc<f16_tag>(plan, ka, st);
    case TFTQ_BF16: return launch_qc<bf16_tag>(plan, ka, st);
    default: return TFTQ_E_DTYPE;
    }
}
