// k_reduce: fused_reduce_fp8 on gfx950.  One .hip file per flavour of the kernel instantiates
// reduce_flavour (below), so that they are compiled side by side.
//
// Follows torchft/quantization.py:261-428 (kernels); design notes in tftq_device.h.

#pragma once

#include "tftq_device.h"

// ---------------------------------------------------------------------------
// reduce
// ---------------------------------------------------------------------------
// The new codes of the register-resident rows leave with streaming stores.  A group of 4
// peers writes a fifth of its traffic, and plain stores left that much dirty in the caches:
// on the fp32 pseudo-gradient of a 1.1 B-parameter model (ws = 4) the kernel took 257 us with
// plain and 215 us with streaming stores, and the dequantize launch behind it 913 against
// 880 us; a group of 8 (a ninth of the traffic) measures the same either way, and so does the
// 4-byte store of the new scale, which stays a plain one.
#define STORE_CODES(val, ptr) STORE_STREAM((val), (ptr))
// Loads dwords [d0, d0+4) of a row payload (ndw dwords long); dwords past the
// end read as 0 and are never touched in memory.  Codes past column n inside
// the last dword are cleared: the reference masks them (:420-424).
DEV u32x4 load_codes(GLOBAL const u32 *payload, int d0, int ndw, int n)
{
    u32x4 w = {0, 0, 0, 0};
    const int rem = ndw - d0;
    if (rem >= 4) {
        w = *(GLOBAL const u32x4_a4 *)(payload + d0);
    } else if (rem > 0) {
        w.x = payload[d0];
        if (rem > 1) w.y = payload[d0 + 1];
        if (rem > 2) w.z = payload[d0 + 2];
    }
    if (n & 3) {
        const int last = ndw - 1 - d0;
        const u32 mask = (1u << (8 * (n & 3))) - 1u;
        if (last == 0) w.x &= mask;
        if (last == 1) w.y &= mask;
        if (last == 2) w.z &= mask;
        if (last == 3) w.w &= mask;
    }
    return w;
}

DEV void store_codes(GLOBAL u32 *payload, int d0, int ndw, const u32x4 w)
{
    const int rem = ndw - d0;
    if (rem >= 4) {
        *(GLOBAL u32x4_a4 *)(payload + d0) = w;
    } else if (rem > 0) {
        payload[d0] = w.x;
        if (rem > 1) payload[d0 + 1] = w.y;
        if (rem > 2) payload[d0 + 2] = w.z;
    }
}

// acc[e] += code[e] / s for the 16 codes of w, s given as (r, r_lo).
// FIRST: acc[e] = code[e] / s, for the first peer of a row.  The reference starts from
// zeros (:405) and 0 + q is q for every q but -0, so the sums can only differ when every
// peer contributes -0: then this sum is -0 where the reference has +0.  requant16 makes
// up for that (a negative zero sum is encoded as +0); the row maximum does not see it.
template <bool FIRST = false>
DEV void accumulate16(float (&acc)[16], const u32x4 w, float r, float r_lo)
{
    const u32 ww[4] = {w.x, w.y, w.z, w.w};

#pragma unroll
    for (int t = 0; t < 4; t++) {
        float f[4];
        unpack_fp8x4(ww[t], f);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float q = div_fast(f[e], r, r_lo);
            acc[4 * t + e] = FIRST ? q : acc[4 * t + e] + q;
        }
    }
}

// (acc * s2) / div, left to right (:364).  Without GDIV, inv_div (1 for SUM) is
// the exact inverse of a power of two and multiplying by it is the same
// correctly rounded result.  GDIV: div is not a power of two.  For div < 1024
// the quotient comes from inv_div = RN(1 / div) in three operations,
//     q0 = y * inv_div,  rem = fma(-q0, div, y),  q = fma(rem, inv_div, q0),
// which equals RN(y / div) for every binary32 y whose quotient is not close to
// the subnormal range (tests/exact_quotient.c checks all 2^23 mantissas of y
// against every odd div below 1024; powers of two in div only move exponents).
// Below 2^-100 the steps may round differently, but every |q| < 2^-10 gives the
// code +-0, with the sign of y restored by the copysign (-0 / div = -0).
// IEEE: the plain divide, for larger group sizes (div_mode 3).
template <bool GDIV, bool IEEE = false>
DEV float scale_div(float a, float s2, const KCall &p)
{
    const float y = __builtin_fmaf(a, s2, 0.0f);  // a * s2, and +0 for a sum of -0 (see accumulate16)
    if (!GDIV) return y * p.inv_div;
    if (IEEE) return y / p.div;
    const float q0 = y * p.inv_div;
    const float rem = __builtin_fmaf(-q0, p.div, y);
    return __builtin_copysignf(__builtin_fmaf(rem, p.inv_div, q0), y);
}

// row maximum / div (:340); for a power-of-two div the multiplication by the
// exact inverse is the same correctly rounded value, subnormal results included
template <bool GDIV>
DEV float amax_div(float amax, const KCall &p)
{
    return GDIV ? amax / p.div : amax * p.inv_div;
}

template <bool GDIV>
DEV u32x4 requant16(const float (&a)[16], float s2, const KCall &p)
{
    float y[16];
    // Power-of-two div: s2 * inv_div is exact unless it is subnormal, and then
    // a * (s2 * inv_div) rounds the same exact product as (a * s2) * inv_div does in two
    // steps; the two can only differ below 2^-126, where every code is zero anyway.
    const float sf = s2 * p.inv_div;
    const bool fold = !GDIV && (sf == 0.0f || __builtin_fabsf(sf) >= 1.17549435e-38f);
    if (__builtin_amdgcn_ballot_w64(!fold) == 0) {  // one code path per wavefront
#pragma unroll
        for (int e = 0; e < 16; e++) y[e] = __builtin_fmaf(a[e], sf, 0.0f);  // a * sf, and +0 for a sum of -0
    } else {
#pragma unroll
        for (int e = 0; e < 16; e++) y[e] = scale_div<GDIV>(a[e], s2, p);
    }
    u32x4 o;
    o.x = pack_fp8x4(y[0], y[1], y[2], y[3]);
    o.y = pack_fp8x4(y[4], y[5], y[6], y[7]);
    o.z = pack_fp8x4(y[8], y[9], y[10], y[11]);
    o.w = pack_fp8x4(y[12], y[13], y[14], y[15]);
    return o;
}

DEV GLOBAL const u32 *peer_row(const KCall &p, int k, int64_t off)
{
    int peer = p.rank + k;  // :407
    if (peer >= p.ws) peer -= p.ws;

    return as_global<const u32>(p.packed + (int64_t)peer * p.slot_size + off);
}

DEV float guarded_scale(GLOBAL const u32 *prow)
{
    const float sc = as_f(prow[0]);
    return sc == 0.0f ? 1.0f : sc;  // padding rows (:419)
}

// One column at a time with plain IEEE divides, two passes: the path of rows
// in which some peer's scale is outside the range of the fast exact division,
// and of rows too long for registers.  Small code, not tuned.
template <int TEAM, bool GDIV, bool IEEE = false>
DEV void reduce_row_slow(const Seg &s, const KCall &p, int j, int lane, float *lds)
{
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;
    GLOBAL uint8_t *orow = as_global<uint8_t>(p.packed + (int64_t)p.rank * p.slot_size + off);
    float amax = 0.0f, s2 = 0.0f;
#pragma nounroll
    for (int pass = 0; pass < 2; pass++) {
#pragma nounroll
        for (int c = lane; c < s.n; c += TEAM) {
            float a = 0.0f;
#pragma nounroll
            for (int k = 0; k < p.ws; k++) {
                GLOBAL const u32 *prow = peer_row(p, k, off);
                const float sc = guarded_scale(prow);
                const int code = ((GLOBAL const uint8_t *)prow)[4 + c];
                a = a + __builtin_amdgcn_cvt_f32_fp8(code, 0) / sc;
            }
            if (pass == 0) {
                amax = fmaxf(amax, __builtin_fabsf(a));
            } else {
                const float y = scale_div<GDIV, IEEE>(a, s2, p);
                orow[4 + c] = (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(y, 0.0f, 0, false) & 0xFF);
            }
        }
        if (pass == 0) {
            amax = team_max<TEAM>(amax, lds);
            s2 = calc_scale(amax_div<GDIV>(amax, p));
        }
    }
    // the own slot's old scale is an input of every lane: write the new one last (:375)
    __threadfence_block();
    if (TEAM == 256) __syncthreads();
    if (lane == 0) *(GLOBAL u32 *)orow = as_u(s2);
}

// Rows longer than a 256-lane team can keep in registers (more than 16384
// columns): two passes over chunks of 1024 dwords, as the reference does for
// every row (:318-372), but with 16-byte loads, the fast exact division and the
// scales read once.  The second pass reads the peer rows again (from the
// caches if they are still there).
// The passes cover the dwords from d0 on.  The caller deals with the dwords before d0:
// `middle` runs between the first pass and the row maximum and returns their maximum (it
// may read the peers' rows, the own slot included: nothing has been stored yet), `between`
// stores them, when the new scale is known and every lane has finished reading for the
// first pass.  c: division coefficients of peer min(lane, ws - 1), all fast.
// PARK: the sums of the first PARK chunks are parked in LDS (parked: PARK * 16 KB) by the
// first pass and taken from there by the second, which then reads no peer for them.
// A step is a chunk's vectors of up to 8 peers; the loads of the next step are in flight
// while the current one is accumulated (53248 bf16 columns, 8 peers: 62.3 us with steps of 4
// peers one after the other, 56.0 us with steps of 8).
constexpr int R_STEP_PEERS = 8;
template <bool GDIV, int PARK, typename Middle, typename Between>
DEV void reduce_row_two_passes(const Seg &s, const KCall &p, int j, int tid, float *lds, const DivCoef &c,
                               int d0, Middle middle, Between between, float *parked = nullptr)
{
    constexpr int CHUNK = 4 * TFTQ_WG;  // dwords
    const int ndw = (s.row_bytes >> 2) - 1;
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;
    const int ws = p.ws;  // <= 64 here
    GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off);
    const u32 tailmask = (s.n & 3) ? (1u << (8 * (s.n & 3))) - 1u : 0xFFFFFFFFu;
    const int nchunks = (ndw - d0 + CHUNK - 1) / CHUNK;
    const int nbatches = (ws + R_STEP_PEERS - 1) / R_STEP_PEERS;  // steps per chunk
    float amax = 0.0f, s2 = 0.0f;

    struct Step {
        u32x4 w[R_STEP_PEERS];
    };
    // loads of batch `bi` of chunk `ci`
    auto issue = [&](Step &dst, int ci, int bi) {
        const int doff = min(d0 + ci * CHUNK + 4 * tid, ndw - 4);  // the last vector ends with the row
#pragma unroll
        for (int b = 0; b < R_STEP_PEERS; b++)
            dst.w[b] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(peer_row(p, min(bi * R_STEP_PEERS + b, ws - 1), off) + 1 + doff));
    };
    // what both passes do with the sums of a chunk
    auto finish = [&](const float (&acc)[16], int ci, int pass) {
        const int d = d0 + ci * CHUNK;
        const int doff = min(d + 4 * tid, ndw - 4);
        if (pass == 0) {
#pragma unroll
            for (int e = 0; e < 16; e++) amax = fmaxf(amax, __builtin_fabsf(acc[e]));
            if (PARK > 0 && ci < PARK) {  // every lane reads back only what it wrote
#pragma unroll
                for (int e = 0; e < 16; e++) parked[(ci * 16 + e) * TFTQ_WG + tid] = acc[e];
            }
        } else {
            // the moved-back last vector overlaps its neighbour, which may sit in another
            // wavefront: nobody stores before everybody has read the own slot's chunk
            __syncthreads();
            if (d + 4 * tid < ndw) {
                const u32x4 o = requant16<GDIV>(acc, s2, p);
                if (doff >= d) {
                    STORE_CODES(o, (GLOBAL u32x4_a4 *)(orow + 1 + doff));
                } else {
                    // The vector reaches back into the dwords before this chunk, whose
                    // codes have already been replaced in the own slot: what was
                    // accumulated for those dwords is meaningless and they are final already.
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (doff + e >= d) orow[1 + doff + e] = o[e];
                }
            }
        }
    };

    auto run_pass = [&](auto pass_c) {
        constexpr int pass = decltype(pass_c)::value;
        float acc[16];
        // the second pass takes the parked chunks from LDS and loads from the first one behind them
        const int first = pass == 0 ? 0 : min(PARK, nchunks);
        if (pass == 1) {
#pragma nounroll
            for (int ci = 0; ci < first; ci++) {
#pragma unroll
                for (int e = 0; e < 16; e++) acc[e] = parked[(ci * 16 + e) * TFTQ_WG + tid];
                finish(acc, ci, 1);
            }
        }
        // steps (chunk, batch) in order; ci, bi: the step to consume, ni, nb: the step to issue
        int ci = first, bi = 0, ni = first, nb = 0;
        auto advance = [&](int &chunk, int &batch) {
            if (++batch == nbatches) {
                batch = 0;
                ++chunk;
            }
        };
        auto consume = [&](const Step &src) {
            const u32 mask = min(d0 + ci * CHUNK + 4 * tid, ndw - 4) == ndw - 4 ? tailmask : 0xFFFFFFFFu;
            if (bi == 0) {
#pragma unroll
                for (int e = 0; e < 16; e++) acc[e] = 0.0f;
            }
#pragma unroll
            for (int b = 0; b < R_STEP_PEERS; b++) {
                const int k = bi * R_STEP_PEERS + b;
                u32x4 w = src.w[b];
                w.w &= mask;
                if (k < ws) accumulate16(acc, w, bcast_lane(c.r, k), bcast_lane(c.r_lo, k));
            }
            if (bi == nbatches - 1) finish(acc, ci, pass);
            advance(ci, bi);
        };
        Step A, B;
        if (ni < nchunks) {
            issue(A, ni, nb);
            advance(ni, nb);
        }
#pragma nounroll
        while (ci < nchunks) {  // A holds the step to consume
            const bool more = ni < nchunks;
            if (more) {
                issue(B, ni, nb);
                advance(ni, nb);
            }
            consume(A);
            if (more) {
                if (ni < nchunks) {
                    issue(A, ni, nb);
                    advance(ni, nb);
                }
                consume(B);
            }
        }
    };
    run_pass(std::integral_constant<int, 0>());
    amax = fmaxf(amax, middle());
    amax = team_max<256>(amax, lds);  // every wavefront has read the old scales by now
    s2 = calc_scale(amax_div<GDIV>(amax, p));
    between(s2);
    run_pass(std::integral_constant<int, 1>());
    if (tid == 0) orow[0] = as_u(s2);  // :375
}

template <bool GDIV>
DEV void reduce_row_long(const Seg &s, const KCall &p, int j, int tid, float *lds)
{
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;
    const DivCoef c = make_div(guarded_scale(peer_row(p, min(tid & 63, p.ws - 1), off)));
    if (__builtin_amdgcn_ballot_w64(!c.fast) != 0) {  // same in the four wavefronts
        reduce_row_slow<256, GDIV>(s, p, j, tid, lds);
        return;
    }
    reduce_row_two_passes<GDIV, 0>(s, p, j, tid, lds, c, 0, [] { return 0.0f; }, [](float) {});
}

// Wide kernel, rows of more than 8192 payload dwords: the sums of the first 8192
// dwords stay in registers (128 per lane), those of the next 4096 are parked in
// 64 KB of LDS and only the rest of the row makes two passes, so the peers are
// read 1 + rest / length times instead of twice (53248 columns: 1.08 times; with 48 KB of
// LDS 1.15 times and 57.3 instead of 53.4 us).  Two workgroups of 64 KB fit the 160 KB of a
// CU, and the registers admit no more than two.
// The part in registers takes its peers through the rolling window of reduce_rows_roll
// (53248 columns: 65.4 -> 62.3 us against all vectors of a peer loaded, then summed).
constexpr int R_PARKED_CHUNKS = 4;  // chunks of 1024 dwords = 16 KB of sums each
template <bool GDIV>
DEV void reduce_row_hybrid(const Seg &s, const KCall &p, int j, int tid, float *lds, float *parked)
{
    constexpr int UNITS = TFTQ_R_DWORDS_WIDE / (4 * TFTQ_WG);  // 8
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;
    const int ws = p.ws;  // <= 64 here
    const DivCoef c = make_div(guarded_scale(peer_row(p, min(tid & 63, ws - 1), off)));
    if (__builtin_amdgcn_ballot_w64(!c.fast) != 0) {  // same in the four wavefronts
        reduce_row_slow<256, GDIV>(s, p, j, tid, lds);
        return;
    }
    // The part of the row behind the registers' makes its first pass first (its loads pipelined in
    // registers that the sums of the part in front do not hold yet), then the part in front
    // is summed, then the row maximum is known and both are stored.
    float acc[UNITS][16];  // set by the first peer
    auto front = [&]() {
        // the rolling window of reduce_rows_roll: vector u of the next peer is loaded as soon as
        // vector u of this one has left its registers
        u32x4 w[UNITS];
        {
            GLOBAL const u32 *pv = peer_row(p, 0, off) + 1;
#pragma unroll
            for (int u = 0; u < UNITS; u++) w[u] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(pv + 4 * (u * TFTQ_WG + tid)));
        }
        {   // the first peer (a group of one reads it a second time and ignores that)
            const float pr = bcast_lane(c.r, 0), pl = bcast_lane(c.r_lo, 0);
            GLOBAL const u32 *pv = peer_row(p, min(1, ws - 1), off) + 1;
#pragma unroll
            for (int u = 0; u < UNITS; u++) {
                u32x4 x = w[u];
                asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w));
                w[u] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(pv + 4 * (u * TFTQ_WG + tid)));
                accumulate16<true>(acc[u], x, pr, pl);
            }
        }
#pragma nounroll
        for (int k = 1; k + 1 < ws; k++) {
            const float pr = bcast_lane(c.r, k), pl = bcast_lane(c.r_lo, k);
            GLOBAL const u32 *pv = peer_row(p, k + 1, off) + 1;
#pragma unroll
            for (int u = 0; u < UNITS; u++) {
                u32x4 x = w[u];
                asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w));  // taken out before the registers are loaded again
                w[u] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(pv + 4 * (u * TFTQ_WG + tid)));
                accumulate16(acc[u], x, pr, pl);
            }
        }
        if (ws > 1) {
            const float pr = bcast_lane(c.r, ws - 1), pl = bcast_lane(c.r_lo, ws - 1);
#pragma unroll
            for (int u = 0; u < UNITS; u++) accumulate16(acc[u], w[u], pr, pl);
        }
        float amax = 0.0f;
#pragma unroll
        for (int u = 0; u < UNITS; u++)
#pragma unroll
            for (int e = 0; e < 16; e++) amax = fmaxf(amax, __builtin_fabsf(acc[u][e]));
        return amax;
    };
    GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off);
    reduce_row_two_passes<GDIV, R_PARKED_CHUNKS>(s, p, j, tid, lds, c, TFTQ_R_DWORDS_WIDE, front, [&](float s2) {
#pragma unroll
        for (int u = 0; u < UNITS; u++)
            STORE_CODES(requant16<GDIV>(acc[u], s2, p), (GLOBAL u32x4_a4 *)(orow + 1 + 4 * (u * TFTQ_WG + tid)));
    }, parked);
}

// Register-resident row: the team holds all accumulators of the row, each peer
// row is read once.  UNITS = 16-byte vectors of codes per lane and peer.  Teams of 64 and 256 lanes
// in groups of more than 64 peers.
template <int TEAM, int UNITS, bool GDIV>
DEV void reduce_row(const Seg &s, const KCall &p, int j, int lane, float *lds)
{
    constexpr int PB = 8 / UNITS;  // peers whose loads are in flight together
    if (j >= s.slice_rows) return;  // a team leaves whole: its lanes share the row
    const int ndw = (s.row_bytes >> 2) - 1;
    const int n = s.n;
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;
    const int wlane = threadIdx.x & 63;

    float acc[UNITS][16];
#pragma unroll
    for (int u = 0; u < UNITS; u++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[u][e] = 0.0f;

    for (int kc = 0; kc < p.ws; kc += 64) {
        const int kend = min(p.ws, kc + 64);
        // Wide teams: lane l of every wavefront fetches the scale of peer kc + l
        // first, then the codes of the first peers go in flight, and only then
        // are the scales turned into division coefficients.
        float my_scale = 1.0f;
        if (kc + wlane < p.ws) my_scale = guarded_scale(peer_row(p, kc + wlane, off));

        u32x4 w[PB][UNITS];
        auto load_batch = [&](int k0) {
#pragma unroll
            for (int b = 0; b < PB; b++) {
                if (k0 + b < kend) {
                    GLOBAL const u32 *prow = peer_row(p, k0 + b, off);
#pragma unroll
                    for (int u = 0; u < UNITS; u++)
                        w[b][u] = load_codes(prow + 1, (u * TEAM + lane) * 4, ndw, n);
                }
            }
        };
        load_batch(kc);

        float cr = 1.0f, cl = 0.0f;
        {
            const DivCoef c = make_div(my_scale);
            cr = c.r;
            cl = c.r_lo;
            if (__builtin_amdgcn_ballot_w64(!c.fast) != 0) {  // some peer needs the plain divide
                reduce_row_slow<TEAM, GDIV>(s, p, j, lane, lds);
                return;
            }
        }
        for (int k0 = kc; k0 < kend; k0 += PB) {
            if (k0 != kc) load_batch(k0);
#pragma unroll
            for (int b = 0; b < PB; b++) {
                if (k0 + b < kend) {
                    const float pr = bcast_lane(cr, k0 + b - kc), pl = bcast_lane(cl, k0 + b - kc);
#pragma unroll
                    for (int u = 0; u < UNITS; u++) accumulate16(acc[u], w[b][u], pr, pl);
                }
            }
        }
    }

    float amax = 0.0f;
#pragma unroll
    for (int u = 0; u < UNITS; u++)
#pragma unroll
        for (int e = 0; e < 16; e++) amax = fmaxf(amax, __builtin_fabsf(acc[u][e]));
    amax = team_max<TEAM>(amax, lds);
    const float s2 = calc_scale(amax_div<GDIV>(amax, p));  // :340

    GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off);
#pragma unroll
    for (int u = 0; u < UNITS; u++)
        store_codes(orow + 1, (u * TEAM + lane) * 4, ndw, requant16<GDIV>(acc[u], s2, p));
    // Every lane read the old scale of the own slot before team_max (wide
    // teams synchronise there; narrow teams are one wavefront in program order).
    if (lane == 0) orow[0] = as_u(s2);  // :375
}

// One row per team, software-pipelined over the peers: the codes of the next
// batch of peers are in flight while the current batch is accumulated.  A
// batch is R_VPB 16-byte vectors per lane: R_VPB / UNITS peers.  Loads carry no
// branch: a lane past the end of the row re-reads the row's last vector, a
// batch past the last peer re-reads the last peer, and both are ignored later.
// Needs ws <= min(TEAM, 64) (lane l of a team, or of each of its wavefronts,
// holds the scale of peer l) and rows of at least one 16-byte vector.  A team
// whose row is past the end (`valid` false) is given the last row and stores
// nothing, so that the wavefront stays converged for the cross-lane operations.
// (Several rows per team with prefetch of the next row were slower for every
// row length: independent workgroups keep more loads in flight.)
constexpr int R_VPB = 4;

template <int TEAM, int UNITS, bool PIPE, bool GDIV, int WS = 0>
DEV void reduce_rows(const Seg &s, const KCall &p, int j, int lane, float *lds, bool valid = true)
{
    constexpr int PB = R_VPB / UNITS >= 1 ? R_VPB / UNITS : 1;  // peers per batch
    const int ndw = (s.row_bytes >> 2) - 1;  // >= 4 here
    // WS: the group size when it is known at compile time (the loops over the peers then
    // unroll into straight-line code); 0: p.ws
    const int ws = WS ? WS : p.ws;
    const int nb = (ws + PB - 1) / PB;  // batches
    const int wlane = TEAM >= 64 ? (int)(threadIdx.x & 63u) : lane;
    const int speer = min(wlane, ws - 1);  // the peer whose scale this lane fetches
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;

    // Vector u of this lane starts at dword doff[u].  The last vector of a row whose
    // length is not a multiple of 4 dwords is moved back so that it ends with the row:
    // it overlaps its neighbour, both lanes compute and store the same values.  Lanes
    // past the row's end re-read the last vector and do not store.
    int doff[UNITS];
    u32 padmask[UNITS];  // clears the bytes past column n in the row's last dword (:420-424)
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        doff[u] = min(4 * (u * TEAM + lane), ndw - 4);
        padmask[u] = (doff[u] == ndw - 4 && (s.n & 3)) ? (1u << (8 * (s.n & 3))) - 1u : 0xFFFFFFFFu;
    }

    // lane l: scale of peer min(l, ws - 1), first in the queue of loads
    const float raw_scale = as_f(peer_row(p, speer, off)[0]);

    struct Batch {
        u32x4 w[PB][UNITS];
    };
    Batch A, B;
    auto issue = [&](Batch &dst, int batch) {
#pragma unroll
        for (int b = 0; b < PB; b++) {
            GLOBAL const u32 *pv = peer_row(p, min(batch * PB + b, ws - 1), off) + 1;
#pragma unroll
            for (int u = 0; u < UNITS; u++)
                dst.w[b][u] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(pv + doff[u]));
        }
    };

    issue(A, 0);
    if (PIPE && nb > 1) issue(B, 1);
    // the loads above are issued before anything below: left to itself, the scheduler moves
    // them down between the accumulation steps of the straight-line variants
    __builtin_amdgcn_sched_barrier(0);

    const float sc = raw_scale == 0.0f ? 1.0f : raw_scale;  // padding rows (:419)
    const DivCoef c = make_div(sc);
    if (__builtin_amdgcn_ballot_w64(!c.fast) != 0) {  // same in all wavefronts of the team
        if (valid) reduce_row_slow<TEAM, GDIV>(s, p, j, lane, lds);  // some peer needs the plain divide
        return;
    }

    float acc[UNITS][16];  // set by the first peer
    auto consume = [&](const Batch &src, int batch, auto first_c) {
        constexpr bool FIRST = decltype(first_c)::value;
#pragma unroll
        for (int b = 0; b < PB; b++) {
            const int k = batch * PB + b;
            if (k < ws) {
                const float pr = team_bcast<TEAM>(c.r, k), pl = team_bcast<TEAM>(c.r_lo, k);
#pragma unroll
                for (int u = 0; u < UNITS; u++) {
                    u32x4 w = src.w[b][u];
                    w.w &= padmask[u];  // here, not at the load: the load must stay in flight
                    if (FIRST && b == 0) accumulate16<true>(acc[u], w, pr, pl);
                    else accumulate16<false>(acc[u], w, pr, pl);
                }
            }
            // peer after peer: work of later peers that is moved up here only holds registers
            if (WS) __builtin_amdgcn_sched_barrier(0);
        }
    };
    const std::true_type first;
    const std::false_type later;

    consume(A, 0, first);
    if (!PIPE) {  // long rows: one batch in flight keeps the register count down
#pragma nounroll
        for (int i = 1; i < nb; i++) {
            issue(A, i);
            consume(A, i, later);
        }
    } else if (WS) {  // straight-line code: batch i in B for odd i, in A for even i
#pragma unroll
        for (int i = 1; i < (WS + PB - 1) / PB; i++) {
            if (i + 1 < (WS + PB - 1) / PB) {
                issue((i & 1) ? A : B, i + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            consume((i & 1) ? B : A, i, later);
        }
    } else {
#pragma nounroll
        for (int i = 1; i < nb; i += 2) {  // B holds batch i
            if (i + 1 < nb) issue(A, i + 1);
            consume(B, i, later);
            if (i + 1 < nb) {
                if (i + 2 < nb) issue(B, i + 2);
                consume(A, i + 1, later);
            }
        }
    }

    float amax = 0.0f;  // duplicates held by lanes past the row's end do not change it
#pragma unroll
    for (int u = 0; u < UNITS; u++)
#pragma unroll
        for (int e = 0; e < 16; e++) amax = fmaxf(amax, __builtin_fabsf(acc[u][e]));
    amax = team_max<TEAM>(amax, lds);
    const float s2 = calc_scale(amax_div<GDIV>(amax, p));  // :340
    GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off);
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        const u32x4 o = requant16<GDIV>(acc[u], s2, p);
        if (valid && 4 * (u * TEAM + lane) < ndw) STORE_CODES(o, (GLOBAL u32x4_a4 *)(orow + 1 + doff[u]));
    }
    if (valid && lane == 0) orow[0] = as_u(s2);  // :375; all lanes read the old scale before team_max
}

// Rows of one vector per lane and peer in groups of more than 8 peers: the vectors of WINDOW (12 or 16)
// peers are in flight at any time; as soon as a peer's has been taken out of its registers, that of the
// peer WINDOW further on is loaded into them (reduce_rows has 8 in flight and waits for 4 at a time).
// 64 MB of packed bf16 rows, 16 peers: 4096 columns 19.1 -> 16.1 us (4.2 TB/s), 512 columns 18.8 -> 15.9,
// 32 peers 4096 columns 17.2 -> 15.9; a few rows, where the loads' latency is all there is: 32 and 64 peers
// 11.1 -> 7.9 and 19.5 -> 12.5.  A window longer than the group loads its last peer again for nothing:
// with 16 in place of 12, 256 MB of 4096 columns, 9 and 24 peers 61.8 -> 64.8 and 53.8 -> 56.3.
// Requirements as in reduce_rows.
template <int TEAM, int WINDOW, bool GDIV>
DEV void reduce_rows_window(const Seg &s, const KCall &p, int j, int lane, float *lds, bool valid = true)
{
    // the marker keeps the compiler from moving the loads that the two windows have in common in front
    // of the branch between them (48 registers, which it then spills)
    if constexpr (WINDOW == 12) asm volatile("; window of 12");
    const int ndw = (s.row_bytes >> 2) - 1;  // >= 4 here
    const int ws = p.ws;
    const int wlane = TEAM >= 64 ? (int)(threadIdx.x & 63u) : lane;
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;
    const int doff = min(4 * lane, ndw - 4);  // the last vector ends with the row (see reduce_rows)
    const u32 padmask = (doff == ndw - 4 && (s.n & 3)) ? (1u << (8 * (s.n & 3))) - 1u : 0xFFFFFFFFu;

    const float raw_scale = as_f(peer_row(p, min(wlane, ws - 1), off)[0]);
    u32x4 w[WINDOW];
    auto issue = [&](int i, int k) { w[i] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(peer_row(p, min(k, ws - 1), off) + 1 + doff)); };
#pragma unroll
    for (int i = 0; i < WINDOW; i++) issue(i, i);
    __builtin_amdgcn_sched_barrier(0);  // all loads are issued before anything below

    const DivCoef c = make_div(raw_scale == 0.0f ? 1.0f : raw_scale);  // padding rows (:419)
    if (__builtin_amdgcn_ballot_w64(!c.fast) != 0) {  // same in all wavefronts of the team
        if (valid) reduce_row_slow<TEAM, GDIV>(s, p, j, lane, lds);  // some peer needs the plain divide
        return;
    }
    float acc[16];
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = 0.0f;
    auto take = [&](int i, int k, auto more_c) {
        const float pr = team_bcast<TEAM>(c.r, k), pl = team_bcast<TEAM>(c.r_lo, k);
        w[i].w &= padmask;
        accumulate16(acc, w[i], pr, pl);
        __builtin_amdgcn_sched_barrier(0);  // peer after peer, and the registers are loaded again behind their last use
        if constexpr (decltype(more_c)::value) issue(i, k + WINDOW);
    };
    int k0 = 0;
    if constexpr (TEAM >= 64) {
#pragma nounroll
        for (; k0 + WINDOW < ws; k0 += WINDOW) {
#pragma unroll
            for (int i = 0; i < WINDOW; i++) take(i, k0 + i, std::true_type());
        }
    }
#pragma unroll
    for (int i = 0; i < WINDOW; i++)
        if (k0 + i < ws) take(i, k0 + i, std::false_type());

    float amax = 0.0f;  // duplicates held by lanes past the row's end do not change it
#pragma unroll
    for (int e = 0; e < 16; e++) amax = fmaxf(amax, __builtin_fabsf(acc[e]));
    amax = team_max<TEAM>(amax, lds);
    const float s2 = calc_scale(amax_div<GDIV>(amax, p));  // :340
    GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off);
    const u32x4 o = requant16<GDIV>(acc, s2, p);
    if (valid && 4 * lane < ndw) STORE_CODES(o, (GLOBAL u32x4_a4 *)(orow + 1 + doff));
    if (valid && lane == 0) orow[0] = as_u(s2);  // :375; all lanes read the old scale before team_max
}

// Rows of up to 16 * TEAM bytes of codes in teams of 1, 2 or 4 lanes: one vector per lane and
// peer, groups of up to MAXWS (2, 4, 8, 12 or 16) peers, every load of the row in flight at once.  (One
// lane per row reads such a row with two or four loads that lie a row apart from its
// neighbours'; here a load instruction of a wavefront covers 32 or 16 neighbouring rows.)
// Lane l of a team fetches the scales of peers l, l + TEAM, ...: MAXWS / TEAM of them, ahead
// of the codes: a line that a streaming load has brought in is not kept for a later load.
// `valid` as in reduce_rows.
template <int TEAM, int MAXWS, bool GDIV>
DEV void reduce_rows_narrow(const Seg &s, const KCall &p, int j, int lane, float *lds, bool valid)
{
    static_assert(MAXWS <= TEAM || MAXWS % TEAM == 0, "every peer's scale has a lane");
    constexpr int NS = MAXWS > TEAM ? MAXWS / TEAM : 1;  // scales per lane
    const int ndw = (s.row_bytes >> 2) - 1;  // >= 4 here
    const int ws = p.ws;                     // <= MAXWS
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;
    const int doff = min(4 * lane, ndw - 4);  // the last vector ends with the row (see reduce_rows)
    const u32 padmask = (doff == ndw - 4 && (s.n & 3)) ? (1u << (8 * (s.n & 3))) - 1u : 0xFFFFFFFFu;

    float raw[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) raw[i] = as_f(peer_row(p, min(lane + i * TEAM, ws - 1), off)[0]);
    u32x4 w[MAXWS];
#pragma unroll
    for (int k = 0; k < MAXWS; k++)
        w[k] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(peer_row(p, min(k, ws - 1), off) + 1 + doff));
    __builtin_amdgcn_sched_barrier(0);  // all loads are issued before anything below

    DivCoef c[NS];
    bool fast = true;
#pragma unroll
    for (int i = 0; i < NS; i++) {
        c[i] = make_div(raw[i] == 0.0f ? 1.0f : raw[i]);  // padding rows (:419)
        fast = fast && c[i].fast;
    }
    if (__builtin_amdgcn_ballot_w64(!fast) != 0) {
        if (valid) reduce_row_slow<TEAM, GDIV>(s, p, j, lane, lds);  // some peer needs the plain divide
        return;
    }

    float acc[16];  // set by the first peer
#pragma unroll
    for (int k = 0; k < MAXWS; k++) {
        if (k < ws) {
            const float pr = team_bcast<TEAM>(c[k / TEAM].r, k % TEAM);
            const float pl = team_bcast<TEAM>(c[k / TEAM].r_lo, k % TEAM);
            u32x4 v = w[k];
            v.w &= padmask;
            if (k == 0) accumulate16<true>(acc, v, pr, pl);
            else accumulate16<false>(acc, v, pr, pl);
        }
    }

    float amax = 0.0f;  // duplicates held by lanes past the row's end do not change it
#pragma unroll
    for (int e = 0; e < 16; e++) amax = fmaxf(amax, __builtin_fabsf(acc[e]));
    amax = team_max<TEAM>(amax, lds);
    const float s2 = calc_scale(amax_div<GDIV>(amax, p));  // :340
    GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off);
    const u32x4 o = requant16<GDIV>(acc, s2, p);
    if (valid && 4 * lane < ndw) STORE_CODES(o, (GLOBAL u32x4_a4 *)(orow + 1 + doff));
    if (valid && lane == 0) orow[0] = as_u(s2);  // :375; all lanes read the old scale before team_max
}

// One or two peers: four rows of a team at once (tftq_reduce_rows_side), one vector per lane and
// peer, the loads of all rows issued together: 8 per lane, where a row alone has 2.
// Rows j0, j0 + step, ...: neighbouring teams' rows are neighbours.  The sums of one row at a time
// are in registers.  Rows past the end of the tensor are given the last row and store nothing.
template <int TEAM, bool GDIV>
DEV void reduce_rows_side(const Seg &s, const KCall &p, int j0, int step, int lane, float *lds)
{
    constexpr int ROWS = TFTQ_R_SIDE_ROWS, PEERS = 2, N = ROWS * PEERS, NS = N > TEAM ? N / TEAM : 1;  // scales per lane
    const int ndw = (s.row_bytes >> 2) - 1;  // >= 4 here
    const int ws = p.ws;
    const int doff = min(4 * lane, ndw - 4);  // the last vector ends with the row (see reduce_rows)
    const u32 padmask = (doff == ndw - 4 && (s.n & 3)) ? (1u << (8 * (s.n & 3))) - 1u : 0xFFFFFFFFu;
    auto row_off = [&](int r) { return s.slot_off + (int64_t)min(j0 + r * step, s.slice_rows - 1) * s.row_bytes; };

    float raw[NS];  // scale number r * PEERS + k, of row r and peer k, in lane (number % TEAM)
#pragma unroll
    for (int q = 0; q < NS; q++) {
        const int i = lane % N + q * TEAM;
        raw[q] = as_f(peer_row(p, min(i % PEERS, ws - 1), row_off(i / PEERS))[0]);
    }
    u32x4 w[ROWS][PEERS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const int64_t off = row_off(r);
#pragma unroll
        for (int k = 0; k < PEERS; k++)
            w[r][k] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(peer_row(p, min(k, ws - 1), off) + 1 + doff));
    }
    __builtin_amdgcn_sched_barrier(0);  // all loads are issued before anything below

    DivCoef c[NS];
    bool fast = true;
#pragma unroll
    for (int q = 0; q < NS; q++) {
        c[q] = make_div(raw[q] == 0.0f ? 1.0f : raw[q]);  // padding rows (:419)
        fast = fast && c[q].fast;
    }
    if (__builtin_amdgcn_ballot_w64(!fast) != 0) {  // some peer of some row needs the plain divide
#pragma nounroll
        for (int r = 0; r < ROWS; r++)
            if (j0 + r * step < s.slice_rows) reduce_row_slow<TEAM, GDIV>(s, p, j0 + r * step, lane, lds);
        return;
    }
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        float acc[16];  // set by the first peer
#pragma unroll
        for (int k = 0; k < PEERS; k++) {
            if (k < ws) {
                const int i = r * PEERS + k;
                const float pr = team_bcast<TEAM>(c[i / TEAM].r, i % TEAM), pl = team_bcast<TEAM>(c[i / TEAM].r_lo, i % TEAM);
                u32x4 v = w[r][k];
                v.w &= padmask;
                if (k == 0) accumulate16<true>(acc, v, pr, pl);
                else accumulate16<false>(acc, v, pr, pl);
            }
        }
        float amax = 0.0f;  // duplicates held by lanes past the row's end do not change it
#pragma unroll
        for (int e = 0; e < 16; e++) amax = fmaxf(amax, __builtin_fabsf(acc[e]));
        amax = team_max<TEAM>(amax, lds);
        const float s2 = calc_scale(amax_div<GDIV>(amax, p));  // :340
        const bool valid = j0 + r * step < s.slice_rows;
        GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + row_off(r));
        const u32x4 o = requant16<GDIV>(acc, s2, p);
        if (valid && 4 * lane < ndw) STORE_CODES(o, (GLOBAL u32x4_a4 *)(orow + 1 + doff));
        if (valid && lane == 0) orow[0] = as_u(s2);  // :375; all loads of the row came before
    }
}

// The rows of a wavefront's teams, side by side; false when the tensor's rows go one at a time.
template <int TEAM, bool GDIV>
DEV bool reduce_side(const Seg &s, const KCall &p, int blk, int tid, float *lds)
{
    constexpr int TW = 64 / TEAM;  // teams per wavefront
    if (s.side == 1) return false;  // same for all
    const int first = (blk * 4 + __builtin_amdgcn_readfirstlane(tid >> 6)) * TW * TFTQ_R_SIDE_ROWS;
    if (first >= s.slice_rows) return true;  // the whole wavefront leaves
    const int j0 = first + (tid & 63) / TEAM;
    reduce_rows_side<TEAM, GDIV>(s, p, j0, TW, tid % TEAM, lds);
    return true;
}

// Rows of up to 16 * TEAM bytes of codes in groups of more peers than a team (or the registers)
// holds at once: one vector per lane and peer, R_CHUNK peers at a time, the next chunk's scales
// and codes in flight while the current one is accumulated.  Lane l of a team fetches the scales
// of the chunk's peers l, l + TEAM, ...  As everywhere in this file the loads carry no branch.
// (A load under a condition waits for the one before it: with such loads a row cost its team a
// trip to memory per peer, and a list whose tensors have a few rows each, so that one wavefront
// does a whole tensor, waits for exactly that.  10 000 tensors of up to 4096 elements, 16 peers:
// 60.1 -> 36.1 us, of that reduce_col1_few about half.  24 peers, 60 columns: 32 -> 12.5 us.)
// `valid` as in reduce_rows.
constexpr int R_CHUNK = 8;
template <int TEAM, bool GDIV>
DEV void reduce_rows_chunks(const Seg &s, const KCall &p, int j, int lane, float *lds, bool valid)
{
    constexpr int CH = TEAM == 1 ? R_CHUNK / 2 : R_CHUNK;  // a lane alone holds the coefficients of all of them
    constexpr int NS = CH > TEAM ? CH / TEAM : 1;  // scales per lane
    const int ndw = (s.row_bytes >> 2) - 1;  // >= 4 here
    const int ws = p.ws;
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;
    const int doff = min(4 * lane, ndw - 4);  // the last vector ends with the row (see reduce_rows)
    const u32 padmask = (doff == ndw - 4 && (s.n & 3)) ? (1u << (8 * (s.n & 3))) - 1u : 0xFFFFFFFFu;

    struct Chunk {
        float raw[NS];
        u32x4 w[CH];
    };
    auto issue = [&](Chunk &c, int k0) {
#pragma unroll
        for (int i = 0; i < NS; i++) c.raw[i] = as_f(peer_row(p, min(k0 + lane % CH + i * TEAM, ws - 1), off)[0]);
#pragma unroll
        for (int k = 0; k < CH; k++)
            c.w[k] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(peer_row(p, min(k0 + k, ws - 1), off) + 1 + doff));
        __builtin_amdgcn_sched_barrier(0);  // all loads are issued before anything below
    };
    float acc[16];
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = 0.0f;
    // false: some peer needs the plain divide (the same for the whole wavefront)
    auto consume = [&](const Chunk &c, int k0) {
        DivCoef d[NS];
        bool fast = true;
#pragma unroll
        for (int i = 0; i < NS; i++) {
            d[i] = make_div(c.raw[i] == 0.0f ? 1.0f : c.raw[i]);  // padding rows (:419)
            fast = fast && d[i].fast;
        }
        if (__builtin_amdgcn_ballot_w64(!fast) != 0) return false;
#pragma unroll
        for (int k = 0; k < CH; k++) {
            if (k0 + k < ws) {
                const float pr = team_bcast<TEAM>(d[k / TEAM].r, k % TEAM);
                const float pl = team_bcast<TEAM>(d[k / TEAM].r_lo, k % TEAM);
                u32x4 v = c.w[k];
                v.w &= padmask;
                accumulate16(acc, v, pr, pl);
            }
        }
        return true;
    };
    Chunk A, B;
    bool fast = true;
    issue(A, 0);
#pragma nounroll
    for (int k0 = 0; k0 < ws; k0 += 2 * CH) {  // A holds the chunk at k0
        if (k0 + CH < ws) issue(B, k0 + CH);
        if (!(fast = consume(A, k0))) break;
        if (k0 + CH < ws) {
            if (k0 + 2 * CH < ws) issue(A, k0 + 2 * CH);
            if (!(fast = consume(B, k0 + CH))) break;
        }
    }
    if (!fast) {
        if (valid) reduce_row_slow<TEAM, GDIV>(s, p, j, lane, lds);
        return;
    }
    float amax = 0.0f;  // duplicates held by lanes past the row's end do not change it
#pragma unroll
    for (int e = 0; e < 16; e++) amax = fmaxf(amax, __builtin_fabsf(acc[e]));
    amax = team_max<TEAM>(amax, lds);
    const float s2 = calc_scale(amax_div<GDIV>(amax, p));  // :340
    GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off);
    const u32x4 o = requant16<GDIV>(acc, s2, p);
    if (valid && 4 * lane < ndw) STORE_CODES(o, (GLOBAL u32x4_a4 *)(orow + 1 + doff));
    if (valid && lane == 0) orow[0] = as_u(s2);  // :375; all lanes read the old scale before team_max
}

// Rows of ND = 1, 2 or 3 payload dwords (2 to 12 columns), a lane per row: the scale and all codes
// of a row come in with one load of ND + 1 dwords, neighbouring lanes' rows are neighbours in
// memory, and the next R_CHUNK peers are in flight while the current ones are accumulated.
// [6291456, 3] bf16 against four clamped dword loads per row and peer: 2 peers 75 -> 35 us,
// 8 peers 27.5 -> 14.3 us; [4194304, 5]: 54.5 -> 28, 23.1 -> 13.8 us.
template <int ND, bool GDIV>
DEV void reduce_rows_tiny(const Seg &s, const KCall &p, int j, float *lds, bool valid)
{
    typedef u32 Row __attribute__((ext_vector_type(ND + 1)));
    typedef Row Row_a4 __attribute__((aligned(4)));
    const int ws = p.ws;
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;
    const u32 padmask = (s.n & 3) ? (1u << (8 * (s.n & 3))) - 1u : 0xFFFFFFFFu;
    struct Chunk {
        Row w[R_CHUNK];
    };
    auto issue = [&](Chunk &c, int k0) {
#pragma unroll
        for (int k = 0; k < R_CHUNK; k++) c.w[k] = LOAD_STREAM((GLOBAL const Row_a4 *)peer_row(p, min(k0 + k, ws - 1), off));
        __builtin_amdgcn_sched_barrier(0);
    };
    float acc[4 * ND];
#pragma unroll
    for (int e = 0; e < 4 * ND; e++) acc[e] = 0.0f;
    auto consume = [&](const Chunk &c, int k0) {
        bool fast = true;
#pragma unroll
        for (int k = 0; k < R_CHUNK; k++) fast = fast && (c.w[k][0] == 0u || scale_is_fast(as_f(c.w[k][0])));
        if (__builtin_amdgcn_ballot_w64(!fast) != 0) return false;
#pragma unroll
        for (int k = 0; k < R_CHUNK; k++) {
            if (k0 + k < ws) {
                const float sc = as_f(c.w[k][0]);
                const DivCoef d = make_div(sc == 0.0f ? 1.0f : sc);  // padding rows (:419)
#pragma unroll
                for (int t = 0; t < ND; t++) {
                    float f[4];
                    unpack_fp8x4(t == ND - 1 ? c.w[k][1 + t] & padmask : c.w[k][1 + t], f);
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[4 * t + e] = acc[4 * t + e] + div_fast(f[e], d.r, d.r_lo);
                }
            }
        }
        return true;
    };
    Chunk A, B;
    bool fast = true;
    issue(A, 0);
#pragma nounroll
    for (int k0 = 0; k0 < ws; k0 += 2 * R_CHUNK) {
        if (k0 + R_CHUNK < ws) issue(B, k0 + R_CHUNK);
        if (!(fast = consume(A, k0))) break;
        if (k0 + R_CHUNK < ws) {
            if (k0 + 2 * R_CHUNK < ws) issue(A, k0 + 2 * R_CHUNK);
            if (!(fast = consume(B, k0 + R_CHUNK))) break;
        }
    }
    if (!fast) {
        if (valid) reduce_row_slow<1, GDIV>(s, p, j, 0, lds);
        return;
    }
    float amax = 0.0f;
#pragma unroll
    for (int e = 0; e < 4 * ND; e++) amax = fmaxf(amax, __builtin_fabsf(acc[e]));
    const float s2 = calc_scale(amax_div<GDIV>(amax, p));  // :340
    Row o;
    o[0] = as_u(s2);
#pragma unroll
    for (int t = 0; t < ND; t++)
        o[1 + t] = pack_fp8x4(scale_div<GDIV>(acc[4 * t], s2, p), scale_div<GDIV>(acc[4 * t + 1], s2, p),
                              scale_div<GDIV>(acc[4 * t + 2], s2, p), scale_div<GDIV>(acc[4 * t + 3], s2, p));
    if (valid) STORE_CODES(o, (GLOBAL Row_a4 *)as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off));
}

// One row per team with UNITS >= 2 vectors per lane and peer, as a rolling window over the
// peers: as soon as a lane has taken vector u of peer k out of its registers, the load of
// vector u of peer k + 1 is issued into them, so UNITS loads are in flight all the time at
// the register cost of one peer.  The last peer is peeled off: nothing is loaded behind it.
// Same requirements as reduce_rows.
template <int TEAM, int UNITS, bool GDIV>
DEV void reduce_rows_roll(const Seg &s, const KCall &p, int j, int lane, float *lds, bool valid = true)
{
    const int ndw = (s.row_bytes >> 2) - 1;  // >= 4 here
    const int ws = p.ws;
    const int wlane = TEAM >= 64 ? (int)(threadIdx.x & 63u) : lane;
    const int speer = min(wlane, ws - 1);  // the peer whose scale this lane fetches
    const int64_t off = s.slot_off + (int64_t)j * s.row_bytes;

    u32 boff[UNITS];     // byte offset of vector u of this lane in the payload (see reduce_rows)
    u32 padmask[UNITS];
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        const int d = min(4 * (u * TEAM + lane), ndw - 4);
        boff[u] = 4u * (u32)d;
        padmask[u] = (d == ndw - 4 && (s.n & 3)) ? (1u << (8 * (s.n & 3))) - 1u : 0xFFFFFFFFu;
    }
    const float raw_scale = as_f(peer_row(p, speer, off)[0]);
    u32x4 w[UNITS];
    {
        GLOBAL const uint8_t *pv = (GLOBAL const uint8_t *)(peer_row(p, 0, off) + 1);
#pragma unroll
        for (int u = 0; u < UNITS; u++) w[u] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(pv + boff[u]));
    }
    float acc[UNITS][16];  // set by the first peer
    const float sc = raw_scale == 0.0f ? 1.0f : raw_scale;  // padding rows (:419)
    const DivCoef c = make_div(sc);
    const bool row_fast = __builtin_amdgcn_ballot_w64(!c.fast) == 0;  // same in all wavefronts of the team
    if (row_fast) {
        {   // the first peer (a group of one reads it a second time and ignores that)
            const float pr = team_bcast<TEAM>(c.r, 0), pl = team_bcast<TEAM>(c.r_lo, 0);
            GLOBAL const uint8_t *pv = (GLOBAL const uint8_t *)(peer_row(p, min(1, ws - 1), off) + 1);
#pragma unroll
            for (int u = 0; u < UNITS; u++) {
                u32x4 x = w[u];
                asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w));
                w[u] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(pv + boff[u]));
                x.w &= padmask[u];
                accumulate16<true>(acc[u], x, pr, pl);
            }
        }
#pragma nounroll
        for (int k = 1; k + 1 < ws; k++) {
            const float pr = team_bcast<TEAM>(c.r, k), pl = team_bcast<TEAM>(c.r_lo, k);
            GLOBAL const uint8_t *pv = (GLOBAL const uint8_t *)(peer_row(p, k + 1, off) + 1);
#pragma unroll
            for (int u = 0; u < UNITS; u++) {
                u32x4 x = w[u];
                asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w));  // taken out before the registers are loaded again
                w[u] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(pv + boff[u]));
                x.w &= padmask[u];
                accumulate16(acc[u], x, pr, pl);
            }
        }
        if (ws > 1) {
            const float pr = team_bcast<TEAM>(c.r, ws - 1), pl = team_bcast<TEAM>(c.r_lo, ws - 1);
#pragma unroll
            for (int u = 0; u < UNITS; u++) {
                u32x4 x = w[u];
                x.w &= padmask[u];
                accumulate16(acc[u], x, pr, pl);
            }
        }
        float amax = 0.0f;  // duplicates held by lanes past the row's end do not change it
#pragma unroll
        for (int u = 0; u < UNITS; u++)
#pragma unroll
            for (int e = 0; e < 16; e++) amax = fmaxf(amax, __builtin_fabsf(acc[u][e]));
        amax = team_max<TEAM>(amax, lds);
        const float s2 = calc_scale(amax_div<GDIV>(amax, p));  // :340
        GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off);
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            const u32x4 o = requant16<GDIV>(acc[u], s2, p);
            if (valid && 4 * (u * TEAM + lane) < ndw) STORE_CODES(o, (GLOBAL u32x4_a4 *)((GLOBAL uint8_t *)(orow + 1) + boff[u]));
        }
        if (valid && lane == 0) orow[0] = as_u(s2);  // :375; all lanes read the old scale before team_max
    } else if (valid) {
        reduce_row_slow<TEAM, GDIV>(s, p, j, lane, lds);  // some peer needs the plain divide
    }
}

// Few peers (ws <= 4): ROWS consecutive rows of one team at once, all loads of
// all rows issued together, so that a lane has 8 vectors in flight although a
// row has only ws * UNITS of them.  ws * UNITS * ROWS <= 8.  Rows past the end of
// the tensor are given the last row and store nothing.  lds: 4 * ROWS floats.
template <int TEAM, int UNITS, int ROWS, bool GDIV>
DEV void reduce_rows_at_once(const Seg &s, const KCall &p, int j0, int lane, float *lds)
{
    constexpr int PEERS = 8 / (UNITS * ROWS);  // ws <= PEERS
    const int ndw = (s.row_bytes >> 2) - 1;    // >= 4 here
    const int ws = p.ws;
    const int wlane = (int)(threadIdx.x & 63u);
    const int speer = min(wlane, ws - 1);  // the peer whose scale this lane fetches

    int doff[UNITS];
    u32 padmask[UNITS];  // as in reduce_rows
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        doff[u] = min(4 * (u * TEAM + lane), ndw - 4);
        padmask[u] = (doff[u] == ndw - 4 && (s.n & 3)) ? (1u << (8 * (s.n & 3))) - 1u : 0xFFFFFFFFu;
    }

    int64_t off[ROWS];
    bool valid[ROWS];
    float raw_scale[ROWS];
    u32x4 w[ROWS][PEERS][UNITS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        valid[r] = j0 + r < s.slice_rows;
        off[r] = s.slot_off + (int64_t)min(j0 + r, s.slice_rows - 1) * s.row_bytes;
        raw_scale[r] = as_f(peer_row(p, speer, off[r])[0]);
    }
#pragma unroll
    for (int r = 0; r < ROWS; r++)
#pragma unroll
        for (int k = 0; k < PEERS; k++) {
            GLOBAL const u32 *pv = peer_row(p, min(k, ws - 1), off[r]) + 1;
#pragma unroll
            for (int u = 0; u < UNITS; u++) w[r][k][u] = LOAD_STREAM((GLOBAL const u32x4_a4 *)(pv + doff[u]));
        }

    float amax[ROWS];
    float acc[ROWS][UNITS][16];
    bool fast[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const float sc = raw_scale[r] == 0.0f ? 1.0f : raw_scale[r];  // padding rows (:419)
        const DivCoef c = make_div(sc);
        fast[r] = __builtin_amdgcn_ballot_w64(!c.fast) == 0;  // same in all wavefronts of the team
#pragma unroll
        for (int u = 0; u < UNITS; u++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[r][u][e] = 0.0f;  // a slow row's sums are not used
        amax[r] = 0.0f;
        if (fast[r]) {
#pragma unroll
            for (int k = 0; k < PEERS; k++) {
                if (k < ws) {
                    const float pr = bcast_lane(c.r, k), pl = bcast_lane(c.r_lo, k);
#pragma unroll
                    for (int u = 0; u < UNITS; u++) {
                        u32x4 v = w[r][k][u];
                        v.w &= padmask[u];
                        if (k == 0) accumulate16<true>(acc[r][u], v, pr, pl);  // the first peer sets the sums
                        else accumulate16(acc[r][u], v, pr, pl);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < UNITS; u++)
#pragma unroll
                for (int e = 0; e < 16; e++) amax[r] = fmaxf(amax[r], __builtin_fabsf(acc[r][u][e]));
        }
    }

    // row maxima over the team: inside the wavefront, then across the four wavefronts
#pragma unroll
    for (int r = 0; r < ROWS; r++) amax[r] = team_max<64>(amax[r], lds);
    if (TEAM == 256) {
        const int wave = threadIdx.x >> 6;
        if (wlane == 0) {
#pragma unroll
            for (int r = 0; r < ROWS; r++) lds[wave * ROWS + r] = amax[r];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ROWS; r++)
            amax[r] = fmaxf(fmaxf(lds[r], lds[ROWS + r]), fmaxf(lds[2 * ROWS + r], lds[3 * ROWS + r]));
        __syncthreads();
    }

#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        if (fast[r]) {
            const float s2 = calc_scale(amax_div<GDIV>(amax[r], p));  // :340
            GLOBAL u32 *orow = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off[r]);
#pragma unroll
            for (int u = 0; u < UNITS; u++) {
                const u32x4 o = requant16<GDIV>(acc[r][u], s2, p);
                if (valid[r] && 4 * (u * TEAM + lane) < ndw) STORE_CODES(o, (GLOBAL u32x4_a4 *)(orow + 1 + doff[u]));
            }
            if (valid[r] && lane == 0) orow[0] = as_u(s2);  // :375
        } else if (valid[r]) {
            reduce_row_slow<TEAM, GDIV>(s, p, j0 + r, lane, lds);  // some peer needs the plain divide
        }
    }
}

// Rows of one column: 8 bytes per row and peer, one plain divide per peer
// (coefficients for the fast division would cost two).
// a += code / scale of a packed row
DEV void accumulate_one(float &a, const u32x2 w)
{
    float sc = as_f(w.x);
    sc = sc == 0.0f ? 1.0f : sc;  // padding rows (:419)
    a = a + __builtin_amdgcn_cvt_f32_fp8((int)w.y, 0) / sc;
}
// [scale, code] of a sum
template <bool GDIV, bool IEEE>
DEV u32x2 requant_one(const KCall &p, float a)
{
    const float s2 = calc_scale(amax_div<GDIV>(fmaxf(0.0f, __builtin_fabsf(a)), p));  // NaN ignored (:331-338)
    u32x2 o;
    o.x = as_u(s2);
    o.y = pack_fp8x4(scale_div<GDIV, IEEE>(a, s2, p), 0.0f, 0.0f, 0.0f) & 0xFFu;
    return o;
}

// At most a row per lane left: the loads of PB peers in flight at once.  (A list of short vectors
// is done when its wavefronts have waited for their peers: 1728 vectors of up to 4096 elements,
// 16 peers: 25.4 us with a peer at a time, 8.6 us with all of them.)
template <int PB, bool GDIV, bool IEEE>
DEV void reduce_col1_few(const Seg &s, const KCall &p, int j, bool valid)
{
    const int64_t off = s.slot_off + (int64_t)j * 8;
    float acc = 0.0f;
#pragma nounroll
    for (int k0 = 0; k0 < p.ws; k0 += PB) {
        u32x2 w[PB];
#pragma unroll
        for (int b = 0; b < PB; b++) w[b] = LOAD_STREAM((GLOBAL const u32x2_a4 *)peer_row(p, min(k0 + b, p.ws - 1), off));
        __builtin_amdgcn_sched_barrier(0);  // all loads are issued before anything below
#pragma unroll
        for (int b = 0; b < PB; b++)
            if (k0 + b < p.ws) accumulate_one(acc, w[b]);
    }
    if (!valid) return;
    const u32x2 o = requant_one<GDIV, IEEE>(p, acc);
    STORE_STREAM(o, (GLOBAL u32x2_a4 *)as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off));
}

// One or two peers: two pairs of neighbouring rows per lane, a pair with one 16-byte access.
// (44 M rows, 2 peers: 92 us with four rows per lane and 8-byte accesses, 86 us.)
template <bool GDIV, bool IEEE>
DEV void reduce_col1_pairs(const Seg &s, const KCall &p, int j0, int tid)
{
    constexpr int PAIRS = 2, PB = 2;
    float acc[PAIRS][2];
    int64_t off[PAIRS];
    u32x4 w[PB][PAIRS];
#pragma unroll
    for (int k = 0; k < PAIRS; k++) {
        acc[k][0] = acc[k][1] = 0.0f;
        // a row without a neighbour (the last of an odd number) comes in behind the one before it
        off[k] = s.slot_off + (int64_t)min(j0 + 2 * (k * TFTQ_WG + tid), s.slice_rows - 2) * 8;
    }
#pragma unroll
    for (int b = 0; b < PB; b++)
#pragma unroll
        for (int k = 0; k < PAIRS; k++) w[b][k] = LOAD_STREAM((GLOBAL const u32x4_a4 *)peer_row(p, min(b, p.ws - 1), off[k]));
    __builtin_amdgcn_sched_barrier(0);  // all loads are issued before anything below
#pragma unroll
    for (int b = 0; b < PB; b++) {
        if (b < p.ws) {
#pragma unroll
            for (int k = 0; k < PAIRS; k++) {
                accumulate_one(acc[k][0], u32x2{w[b][k].x, w[b][k].y});
                accumulate_one(acc[k][1], u32x2{w[b][k].z, w[b][k].w});
            }
        }
    }
#pragma unroll
    for (int k = 0; k < PAIRS; k++) {
        const int j = j0 + 2 * (k * TFTQ_WG + tid);
        if (j >= s.slice_rows) continue;
        const u32x2 a = requant_one<GDIV, IEEE>(p, acc[k][0]), b = requant_one<GDIV, IEEE>(p, acc[k][1]);
        GLOBAL u32 *out = as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off[k]);
        // streaming: neighbouring lanes write neighbouring rows, whole lines per wavefront
        if (j + 1 < s.slice_rows) STORE_STREAM((u32x4{a.x, a.y, b.x, b.y}), (GLOBAL u32x4_a4 *)out);
        else STORE_STREAM(b, (GLOBAL u32x2_a4 *)(out + 2));  // the row before it is another lane's
    }
}

template <bool GDIV, bool IEEE>
DEV void reduce_col1_lane(const Seg &s, const KCall &p, int row)
{
    // a wavefront none of whose lanes has a row leaves at once
    if (__builtin_amdgcn_ballot_w64(row < s.slice_rows) == 0) return;
    const int j = min(row, s.slice_rows - 1);
    if (p.ws <= 4) reduce_col1_few<4, GDIV, IEEE>(s, p, j, row < s.slice_rows);
    else reduce_col1_few<16, GDIV, IEEE>(s, p, j, row < s.slice_rows);
}

// More peers: four rows per lane, a peer at a time (16-byte accesses and two or four peers at a
// time are 2 to 8 % slower from 4 peers on: 33.5 M rows, 8 peers 51.9 us, 54 to 55 us).
// PLAIN: always so (the vectors beside matrices in a layer bucket).
template <bool GDIV, bool IEEE, bool PLAIN>
DEV void reduce_col1(const Seg &s, const KCall &p, int j0, int tid)
{
    if (!PLAIN && s.slice_rows - j0 > TFTQ_WG && p.ws <= 2) {  // same for the whole workgroup, as is the next
        reduce_col1_pairs<GDIV, IEEE>(s, p, j0, tid);
        return;
    }
    // a wavefront none of whose lanes has a row (rows go up with k) leaves at once
    if (__builtin_amdgcn_ballot_w64(j0 + tid < s.slice_rows) == 0) return;
    if (!PLAIN && s.slice_rows - j0 <= TFTQ_WG) {
        reduce_col1_lane<GDIV, IEEE>(s, p, j0 + tid);
        return;
    }
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    int64_t off[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        off[k] = s.slot_off + (int64_t)min(j0 + k * TFTQ_WG + tid, s.slice_rows - 1) * 8;
#pragma nounroll
    for (int kk = 0; kk < p.ws; kk++) {
        u32x2 w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) w[k] = LOAD_STREAM((GLOBAL const u32x2_a4 *)peer_row(p, kk, off[k]));
#pragma unroll
        for (int k = 0; k < 4; k++) accumulate_one(acc[k], w[k]);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (j0 + k * TFTQ_WG + tid < s.slice_rows) {
            const u32x2 o = requant_one<GDIV, IEEE>(p, acc[k]);
            STORE_STREAM(o, (GLOBAL u32x2_a4 *)as_global<u32>(p.packed + (int64_t)p.rank * p.slot_size + off[k]));
        }
    }
}

// The window of reduce_rows_window for rows of one vector per lane, the one of 12 and 16 that loads
// fewer peers for nothing; 0: reduce_rows.  (A team of 32 lanes gains from 13 peers on, [3461, 400] 12 peers
// 8.1 -> 8.7 us, 13 peers 9.2 -> 8.1; more than 16 peers in a team that is no whole wavefront are more than twice
// slower than in reduce_rows, 19.6 against 40.7 us for 64 MB of 512 columns and 24 peers.)
DEV int reduce_window(int team, int ws)
{
    if (ws <= 8 || (team == 32 && ws <= 12) || (team < 64 && ws > 16)) return 0;
    return (ws + 11) / 12 * 12 < (ws + 15) / 16 * 16 ? 12 : 16;
}

// reduce_rows for a team of TEAM lanes with UNITS vectors per lane and peer: groups of 8 and
// of 4 peers run straight-line code (averages over such groups never need GDIV)
#define TFTQ_REDUCE_ROWS(TEAM, UNITS, ...)                                                        \
    do {                                                                                          \
        if (!GDIV && p.ws == 8) reduce_rows<TEAM, UNITS, true, GDIV, GDIV ? 0 : 8>(__VA_ARGS__);  \
        else if (!GDIV && p.ws == 4) reduce_rows<TEAM, UNITS, true, GDIV, GDIV ? 0 : 4>(__VA_ARGS__); \
        else if (UNITS == 1 && TEAM > 8 && reduce_window(TEAM, p.ws) == 16) reduce_rows_window<TEAM, 16, GDIV>(__VA_ARGS__); \
        else if (UNITS == 1 && TEAM > 8 && TEAM != 32 && reduce_window(TEAM, p.ws) == 12) reduce_rows_window<TEAM, 12, GDIV>(__VA_ARGS__); \
        else reduce_rows<TEAM, UNITS, true, GDIV>(__VA_ARGS__);                                   \
    } while (0)

// reduce_rows_narrow for a team of TEAM lanes, for the smallest of 2, 4, 8, 12 and 16 peers that
// holds the group (a variant for more peers loads the last peer again in their place: averages over 9
// and 12 peers, [2097152, 60], with the variant for 16 33.0 and 31.3 us, for 12 29.7 and 28.9);
// larger groups go through the rows in chunks
#define TFTQ_REDUCE_NARROW(TEAM, ...)                                             \
    do {                                                                          \
        if (p.ws <= 2) reduce_rows_narrow<TEAM, 2, GDIV>(__VA_ARGS__);            \
        else if (p.ws <= 4) reduce_rows_narrow<TEAM, 4, GDIV>(__VA_ARGS__);       \
        else if (p.ws <= 8) reduce_rows_narrow<TEAM, 8, GDIV>(__VA_ARGS__);       \
        else if (p.ws <= 12) reduce_rows_narrow<TEAM, 12, GDIV>(__VA_ARGS__);     \
        else if (p.ws <= 16) reduce_rows_narrow<TEAM, 16, GDIV>(__VA_ARGS__);     \
        else reduce_rows_chunks<TEAM, GDIV>(__VA_ARGS__);                         \
    } while (0)

// FLAVOUR: R_ALL, every kind of row; R_WIDE, for lists with rows of more than 16384 columns:
// every kind, twice the registers, half the resident wavefronts; R_LONG, for lists whose rows
// all run in teams of 64 or 256 lanes or have one column (a layer bucket: matrices, norm
// weights, biases): only those kinds.  What
// the compiler makes of one kind's code depends on what else the kernel holds (registers
// kept across the switch, the order of the blocks): with R_LONG the code for the long rows
// of such lists is compiled on its own and does not move when another kind's code changes.
// R_ONE, for lists of one-column tensors (a flat bucket, a list of vectors): few registers, so
// that a SIMD holds all the wavefronts it can.  From 3 peers on that is too many, each with as many
// streams as there are peers; dynamic LDS that nobody uses then holds a CU to four workgroups
// (33.5 M rows, 8 peers: 55.6 us with eight workgroups, 53.0 with six, 52.2 with four, 57.4 with
// three; 16 peers 52.5, 51.6, 46.6, 53.0; before this variant 51.8 and 48.6).
constexpr unsigned R_ONE_LDS = 40000;
enum { R_ALL = 0, R_WIDE = 1, R_LONG = 2, R_ONE = 3 };
template <int FLAVOUR>
DEV int kind_of(int kind)
{
    if (FLAVOUR == R_LONG) return kind == K_GEN64 ? K_GEN64 : kind == K_COL1 ? K_COL1 : K_GEN256;
    return FLAVOUR == R_ONE && kind != K_COL1_FEW ? (int)K_COL1 : kind;
}
template <bool GDIV, int FLAVOUR, typename A>
DEV void reduce_workgroup(const A &args)
{
    constexpr bool FEW = FLAVOUR == R_ALL || FLAVOUR == R_ONE;  // the kind for little work (pick_few_kinds)
    constexpr bool WIDE = FLAVOUR == R_WIDE;
    __shared__ float lds[16];
    __shared__ float parked[WIDE ? R_PARKED_CHUNKS * 16 * TFTQ_WG : 1];  // wide kernel: 64 KB (two workgroups per CU fit)
    Seg s;
    KCall p;
    int blk;
    if (!locate<ST_R>(args, p, s, blk)) return;
    int tid = threadIdx.x;
    if constexpr (std::is_same<A, KTable>::value) {
        if (args.pieces) {
            // blk is a quarter of a workgroup (tftq_reduce_pieces in tftq_internal.h): this wavefront is
            // wavefront blk % 4 of workgroup blk / 4 of its tensor, whatever its neighbours work on
            tid = (blk & 3) * 64 + (tid & 63);
            blk >>= 2;
        }
    }
    const int ndw = (s.row_bytes >> 2) - 1;
    if (GDIV && p.div_mode == 3) {
        // averages over 1024 peers or more, not a power of two: the untuned path with plain divides
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        switch (kind_of<FLAVOUR>(s.kind[ST_R])) {
        case K_GEN256: reduce_row_slow<256, true, true>(s, p, blk, tid, lds); break;
        case K_GEN64:
            if (blk * 4 + wave < s.slice_rows) reduce_row_slow<64, true, true>(s, p, blk * 4 + wave, tid & 63, lds);
            break;
        case K_GEN32:
            if (blk * 8 + (tid >> 5) < s.slice_rows) reduce_row_slow<32, true, true>(s, p, blk * 8 + (tid >> 5), tid & 31, lds);
            break;
        case K_GEN16:
            if (blk * 16 + (tid >> 4) < s.slice_rows) reduce_row_slow<16, true, true>(s, p, blk * 16 + (tid >> 4), tid & 15, lds);
            break;
        case K_GEN8:
            if (blk * 32 + (tid >> 3) < s.slice_rows) reduce_row_slow<8, true, true>(s, p, blk * 32 + (tid >> 3), tid & 7, lds);
            break;
        case K_GEN4:
            if (blk * 64 + (tid >> 2) < s.slice_rows) reduce_row_slow<4, true, true>(s, p, blk * 64 + (tid >> 2), tid & 3, lds);
            break;
        case K_GEN2:
            if (blk * 128 + (tid >> 1) < s.slice_rows) reduce_row_slow<2, true, true>(s, p, blk * 128 + (tid >> 1), tid & 1, lds);
            break;
        case K_GEN1:
            if (blk * 256 + tid < s.slice_rows) reduce_row_slow<1, true, true>(s, p, blk * 256 + tid, 0, lds);
            break;
        case K_COL1: reduce_col1<true, true, FLAVOUR == R_LONG>(s, p, blk * tftq_col1_rows_per_wg(ST_R), tid); break;
        case K_COL1_FEW:
            if constexpr (FEW) reduce_col1_lane<true, true>(s, p, blk * TFTQ_WG + tid);
            break;
        default: break;
        }
        return;
    }
    // (R_LONG, R_ONE: a kind that they are launched for, whatever the table says)
    switch (kind_of<FLAVOUR>(s.kind[ST_R])) {
    case K_GEN256: {  // one workgroup per row, or per 2 or 4 rows when the group is small
        const int rows = tftq_reduce_rows_at_once(K_GEN256, ndw, p.ws);
        const int j = blk * rows;
        if (rows == 4) {
            reduce_rows_at_once<256, 1, 4, GDIV>(s, p, j, tid, lds);
        } else if (rows == 2) {
            if (ndw <= 1024) reduce_rows_at_once<256, 1, 2, GDIV>(s, p, j, tid, lds);
            else reduce_rows_at_once<256, 2, 2, GDIV>(s, p, j, tid, lds);
        } else if (WIDE && ndw > TFTQ_R_DWORDS && ndw <= TFTQ_R_DWORDS_WIDE && p.ws <= 64) {
            // vectors per lane and peer that this wavefront needs (see below): 4 to 8
            const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            const int nu = min((ndw + 1023) >> 10, (ndw - 256 * wave + 1023) >> 10);
            if (nu <= 4) reduce_rows_roll<256, 4, GDIV>(s, p, j, tid, lds);
            else if (nu == 5) reduce_rows_roll<256, 5, GDIV>(s, p, j, tid, lds);
            else if (nu == 6) reduce_rows_roll<256, 6, GDIV>(s, p, j, tid, lds);
            else if (nu == 7) reduce_rows_roll<256, 7, GDIV>(s, p, j, tid, lds);
            else reduce_rows_roll<256, 8, GDIV>(s, p, j, tid, lds);
        } else if (ndw > TFTQ_R_DWORDS) {
            if (p.ws > 64) reduce_row_slow<256, GDIV>(s, p, j, tid, lds);
            else if (WIDE && ndw > TFTQ_R_DWORDS_WIDE) reduce_row_hybrid<GDIV>(s, p, j, tid, lds, parked);
            else reduce_row_long<GDIV>(s, p, j, tid, lds);
        } else if (p.ws > 64) {
            if (ndw <= 1024) reduce_row<256, 1, GDIV>(s, p, j, tid, lds);
            else reduce_row<256, 4, GDIV>(s, p, j, tid, lds);
        } else {
            // Vectors per lane and peer that this wavefront needs: lane l of the team holds
            // dwords 4 * (256 * u + l) ..., so the upper wavefronts of a row whose length is
            // not a multiple of 1024 dwords need one vector less than the lower ones
            // (10240 columns: 3, 3, 2, 2 instead of 3 each: 55.0 -> 50.4 us on [20480, 10240]).
            // Every variant passes the team's barriers the same number of times.
            const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            // (at least one: a wavefront past the end of a short row still takes part in the barriers)
            const int nu = max(1, min((ndw + 1023) >> 10, (ndw - 256 * wave + 1023) >> 10));
            if (nu == 1) TFTQ_REDUCE_ROWS(256, 1, s, p, j, tid, lds);
            // rows of three or four vectors per lane run the rolling window in all their wavefronts
            // ([20480, 10240]: 53.5 -> 50.4 us against the pipeline in the upper two); rows of two
            // are faster in the pipeline (5120 columns: 50.9 against 62.1 us)
            else if (nu == 2 && ndw > 2048) reduce_rows_roll<256, 2, GDIV>(s, p, j, tid, lds);
            else if (nu == 2) TFTQ_REDUCE_ROWS(256, 2, s, p, j, tid, lds);
            else if (nu == 3) reduce_rows_roll<256, 3, GDIV>(s, p, j, tid, lds);
            else reduce_rows_roll<256, 4, GDIV>(s, p, j, tid, lds);
        }
        break;
    }
    case K_GEN64: {  // one wavefront per row, or per 2 or 4 rows when the group is small
        const int rows = tftq_reduce_rows_at_once(K_GEN64, ndw, p.ws);
        const int j = (blk * 4 + __builtin_amdgcn_readfirstlane(tid >> 6)) * rows;
        if (j >= s.slice_rows) break;  // the whole wavefront leaves
        if (rows == 4) {
            reduce_rows_at_once<64, 1, 4, GDIV>(s, p, j, tid & 63, lds);
        } else if (rows == 2) {
            if (ndw <= 256) reduce_rows_at_once<64, 1, 2, GDIV>(s, p, j, tid & 63, lds);
            else reduce_rows_at_once<64, 2, 2, GDIV>(s, p, j, tid & 63, lds);
        } else if (p.ws > 64) {
            if (ndw <= 256) reduce_row<64, 1, GDIV>(s, p, j, tid & 63, lds);
            else if (ndw <= 512) reduce_row<64, 2, GDIV>(s, p, j, tid & 63, lds);
            else reduce_row_slow<64, GDIV>(s, p, j, tid & 63, lds);
        } else if (ndw <= 256) {
            TFTQ_REDUCE_ROWS(64, 1, s, p, j, tid & 63, lds);
        } else if (ndw <= 512) {
            TFTQ_REDUCE_ROWS(64, 2, s, p, j, tid & 63, lds);
        } else {
            reduce_rows_roll<64, 3, GDIV>(s, p, j, tid & 63, lds);
        }
        break;
    }
    case K_GEN32:
    case K_GEN16:
    case K_GEN8: {
        // one row per team of 32, 16 or 8 lanes
        auto small = [&](auto team_c) {
            constexpr int TEAM = decltype(team_c)::value;
            const int j = blk * (TFTQ_WG / TEAM) + tid / TEAM;
            if (ndw > 4 * TEAM) {  // three vectors per lane (see pick_reduce_kind)
                if (p.ws <= TEAM) reduce_rows_roll<TEAM, 3, GDIV>(s, p, min(j, s.slice_rows - 1), tid % TEAM, lds, j < s.slice_rows);
                else if (j < s.slice_rows) reduce_row_slow<TEAM, GDIV>(s, p, j, tid % TEAM, lds);
            } else if (reduce_side<TEAM, GDIV>(s, p, blk, tid, lds)) {
            } else if (p.ws <= TEAM) {
                TFTQ_REDUCE_ROWS(TEAM, 1, s, p, min(j, s.slice_rows - 1), tid % TEAM, lds, j < s.slice_rows);
            } else if (TEAM == 8 && p.ws <= 16) {
                reduce_rows_narrow<TEAM, 16, GDIV>(s, p, min(j, s.slice_rows - 1), tid % TEAM, lds, j < s.slice_rows);
            } else {
                reduce_rows_chunks<TEAM, GDIV>(s, p, min(j, s.slice_rows - 1), tid % TEAM, lds, j < s.slice_rows);
            }
        };
        if (s.kind[ST_R] == K_GEN32) small(std::integral_constant<int, 32>());
        else if (s.kind[ST_R] == K_GEN16) small(std::integral_constant<int, 16>());
        else small(std::integral_constant<int, 8>());
        break;
    }
    case K_GEN4: {  // one row per team of 4 lanes
        const int j = blk * 64 + (tid >> 2);
        if (reduce_side<4, GDIV>(s, p, blk, tid, lds)) break;
        TFTQ_REDUCE_NARROW(4, s, p, min(j, s.slice_rows - 1), tid & 3, lds, j < s.slice_rows);
        break;
    }
    case K_GEN2: {  // one row per pair of lanes
        const int j = blk * 128 + (tid >> 1);
        if (reduce_side<2, GDIV>(s, p, blk, tid, lds)) break;
        TFTQ_REDUCE_NARROW(2, s, p, min(j, s.slice_rows - 1), tid & 1, lds, j < s.slice_rows);
        break;
    }
    case K_GEN1: {  // one lane per row
        const int j = blk * 256 + tid, jc = min(j, s.slice_rows - 1);
        const bool valid = j < s.slice_rows;
        if (ndw == 4) TFTQ_REDUCE_NARROW(1, s, p, jc, 0, lds, valid);
        else if (ndw == 3) reduce_rows_tiny<3, GDIV>(s, p, jc, lds, valid);
        else if (ndw == 2) reduce_rows_tiny<2, GDIV>(s, p, jc, lds, valid);
        else if (ndw == 1) reduce_rows_tiny<1, GDIV>(s, p, jc, lds, valid);
        else if (valid) reduce_row_slow<1, GDIV>(s, p, j, 0, lds);  // no columns: a scale
        break;
    }
    case K_COL1: reduce_col1<GDIV, false, FLAVOUR == R_LONG>(s, p, blk * tftq_col1_rows_per_wg(ST_R), tid); break;
    case K_COL1_FEW:
        if constexpr (FEW) reduce_col1_lane<GDIV, false>(s, p, blk * TFTQ_WG + tid);
        break;
    default: break;
    }
}

constexpr int reduce_waves(int flavour) { return flavour == R_WIDE ? 2 : flavour == R_ONE ? 8 : 4; }  // per SIMD
template <typename A, bool GDIV, int FLAVOUR>
__global__ __launch_bounds__(TFTQ_WG, reduce_waves(FLAVOUR)) void k_reduce(const A args)
{
    reduce_workgroup<GDIV, FLAVOUR>(args);
}
template <bool GDIV, int FLAVOUR>
__global__ __launch_bounds__(TFTQ_WG, reduce_waves(FLAVOUR)) void k_reduce_one(TFTQ_ONE_PARAMS)
{
    reduce_workgroup<GDIV, FLAVOUR>(one_of(TFTQ_ONE));
}

// The launch of a flavour; defined in tftq_reduce_<flavour>.hip.
template <int FLAVOUR>
__attribute__((visibility("hidden"))) int reduce_flavour(const KArgs &ka, bool gdiv, unsigned lds_bytes, hipStream_t st);
template <> int reduce_flavour<R_ALL>(const KArgs &ka, bool gdiv, unsigned lds_bytes, hipStream_t st);
template <> int reduce_flavour<R_WIDE>(const KArgs &ka, bool gdiv, unsigned lds_bytes, hipStream_t st);
template <> int reduce_flavour<R_LONG>(const KArgs &ka, bool gdiv, unsigned lds_bytes, hipStream_t st);
template <> int reduce_flavour<R_ONE>(const KArgs &ka, bool gdiv, unsigned lds_bytes, hipStream_t st);

#define TFTQ_REDUCE_FLAVOUR(FLAVOUR)                                                                                   \
    template <>                                                                                                        \
    int reduce_flavour<FLAVOUR>(const KArgs &ka, bool gdiv, unsigned lds_bytes, hipStream_t st)                        \
    {                                                                                                                  \
        return with_args(ka, [&](const auto &args) {                                                                   \
            typedef typename std::decay<decltype(args)>::type A;                                                       \
            if constexpr (std::is_same<A, KOne>::value)                                                                \
                return launch_kernel(gdiv ? k_reduce_one<true, FLAVOUR> : k_reduce_one<false, FLAVOUR>, ka, args,      \
                                     lds_bytes, st);                                                                   \
            else                                                                                                       \
                return launch_kernel(gdiv ? k_reduce<A, true, FLAVOUR> : k_reduce<A, false, FLAVOUR>, ka, args,        \
                                     lds_bytes, st);                                                                   \
        });                                                                                                            \
    }
