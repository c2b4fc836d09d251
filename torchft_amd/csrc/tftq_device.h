// Device helpers and launch plumbing shared by the three kernel files
// (tftq_quantize.hip, tftq_reduce_kernels.h, tftq_dequantize.hip): HIP kernels for
// gfx950 (MI355X) and the compute entry points of the C ABI.
//
// Three stages, one launch each, and a second one in quantize for a list's matrices that are stored
// column by column and large enough:
//   k_quantize<T>, k_quantize_cols<T>  fused_quantize_into_fp8   (torchft/quantization.py:53-162)
//   k_reduce                           fused_reduce_fp8          (:261-428)
//   k_dequantize<T>                    fused_dequantize_from_fp8 (:165-258)
//
// Design (none of it follows the reference's launch shape):
//   * a row is owned by a "team" of 1 to 256 lanes chosen from the row length
//     (so that a lane has about 8 loads of 16 bytes in flight; lanes of very
//     short rows work on several rows); the team loads the row once, keeps it in
//     registers, reduces |x| with DPP inside the wavefront (LDS across the four
//     wavefronts of a 256-lane team) and converts from registers with the
//     packed fp8 converts of gfx950.  Every stage reads HBM once.
//   * a launch covers all the tensors of a call (k_quantize and k_quantize_cols
//     share them between them): a workgroup finds its tensor in a table of 64-byte descriptors (in the kernel arguments for
//     short lists) and branches on the team size stored there.
//   * workgroup ids are remapped so that each of the 8 XCDs works on
//     contiguous pieces of every tensor (neighbouring packed rows share cache
//     lines), in reduce the tensors with the heaviest workgroups first.
//   * division by a row scale is exact IEEE division, computed as
//     fma(f, r, f * r_lo) with r = RN(1/s) and r_lo = RN(fma(-s, r, 1) / s).
//     For the 253 finite e4m3 values f and every binary32 s with exponent in
//     [-64, 64] this equals RN(f / s) bit for bit (checked exhaustively by
//     tests/test_exact_division.py); other scales take the plain divide.
//
// Build flags that matter: -ffp-contract=off (the arithmetic contract is
// separate IEEE multiply / divide / add), packed fp32 ops disabled.

#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "../../include/tftq.h"
#include "tftq_internal.h"

typedef uint32_t u32;
typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
typedef u32x2 u32x2_a4 __attribute__((aligned(4)));
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));  // tensor rows: aligned to the element only
typedef u32 u32_a2 __attribute__((aligned(2)));
typedef u32x2 u32x2_a2 __attribute__((aligned(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

struct bf16_tag {};
struct f16_tag {};

#define DEV __device__ __forceinline__
// Streaming accesses for data that is touched once per kernel (measured on
// MI355X: +10 % read bandwidth over plain loads).
#define LOAD_STREAM(ptr) __builtin_nontemporal_load(ptr)
#define STORE_STREAM(val, ptr) __builtin_nontemporal_store((val), (ptr))
#define GLOBAL __attribute__((address_space(1)))

// Tensor addresses arrive as integers; tell the compiler they are global
// memory so that it emits global_* rather than flat_* accesses.
template <typename P>
DEV GLOBAL P *as_global(uint64_t addr)
{
    return (GLOBAL P *)addr;
}
template <typename P>
DEV GLOBAL P *as_global(const void *ptr)
{
    return (GLOBAL P *)(uint64_t)ptr;
}

DEV float as_f(u32 u) { return __uint_as_float(u); }
DEV u32 as_u(float f) { return __float_as_uint(f); }

// ---------------------------------------------------------------------------
// wavefront / team reductions
// ---------------------------------------------------------------------------
template <int CTRL>
DEV float dpp_mov(float v)
{
    const int x = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false));
}

DEV float bcast_lane(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// v of lane k of the caller's team (k uniform).  Teams of whole wavefronts hold
// the same values in every wavefront and read lane k; smaller teams go through
// the LDS crossbar.
template <int TEAM>
DEV float team_bcast(float v, int k)
{
    if constexpr (TEAM >= 64) {
        return bcast_lane(v, k);
    } else if constexpr (TEAM == 1) {
        return v;
    } else {
        const int base = (int)(threadIdx.x & 63u) & ~(TEAM - 1);
        return __int_as_float(__builtin_amdgcn_ds_bpermute((base + k) << 2, __float_as_int(v)));
    }
}

// max over the TEAM lanes that share a row; every lane of the team gets it.
// lds: 4 floats per workgroup, used by 256-lane teams only.
template <int TEAM>
DEV float team_max(float v, float *lds)
{
    if (TEAM >= 2) v = fmaxf(v, dpp_mov<0xB1>(v));   // quad_perm [1,0,3,2]
    if (TEAM >= 4) v = fmaxf(v, dpp_mov<0x4E>(v));   // quad_perm [2,3,0,1]
    if (TEAM >= 8) v = fmaxf(v, dpp_mov<0x141>(v));  // row_half_mirror
    if (TEAM >= 16) v = fmaxf(v, dpp_mov<0x140>(v));  // row_mirror: all 16 lanes of a row agree
    if (TEAM >= 32) {
        const float a = bcast_lane(v, 0), b = bcast_lane(v, 16);
        const float c = bcast_lane(v, 32), d = bcast_lane(v, 48);
        if (TEAM == 32) v = (threadIdx.x & 32) ? fmaxf(c, d) : fmaxf(a, b);
        else v = fmaxf(fmaxf(a, b), fmaxf(c, d));
    }
    if (TEAM == 256) {
        const int wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0) lds[wave] = v;
        __syncthreads();
        v = fmaxf(fmaxf(lds[0], lds[1]), fmaxf(lds[2], lds[3]));
        __syncthreads();
    }
    return v;
}

// ---------------------------------------------------------------------------
// scalar helpers of the arithmetic contract
// ---------------------------------------------------------------------------
// _kernel_calculate_scale (quantization.py:44-50)
DEV float calc_scale(float row_max)
{
    const float s = 448.0f / row_max;
    return s == __builtin_inff() ? 1.0f : s;
}

// Exact f / s for e4m3 values f (see the file header).
struct DivCoef {
    float s, r, r_lo;
    bool fast;
};

// positive, exponent in [-64, 64]
DEV bool scale_is_fast(float s) { return (as_u(s) - (63u << 23)) < (129u << 23); }

// r_lo = RN(e / s) with e = fma(-s, r, 1), without a second divide: one Newton step on
// e * r gives the correctly rounded quotient for every scale in the fast range
// (tests/exact_division.c compares the two for all 2^23 mantissas); outside that range
// the coefficients are not used.
DEV DivCoef make_div(float s)
{
    DivCoef c;
    c.s = s;
    c.r = 1.0f / s;
    const float e = __builtin_fmaf(-s, c.r, 1.0f);
    const float lo = e * c.r;
    c.r_lo = __builtin_fmaf(__builtin_fmaf(-s, lo, e), c.r, lo);
    c.fast = scale_is_fast(s);
    return c;
}

DEV float div_fast(float f, float r, float r_lo) { return __builtin_fmaf(f, r, f * r_lo); }

// Same, with the sign of a zero numerator kept (-0 / s = -0 for s > 0; the fma
// form gives +0).  The sum in reduce cannot tell the two zeros apart, the
// stored result of dequantize can.
DEV float div_fast_signed(float f, float r, float r_lo)
{

    return __builtin_copysignf(div_fast(f, r, r_lo), f);
}

// four e4m3 codes -> four floats
DEV void unpack_fp8x4(u32 w, float (&f)[4])
{
    const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
    const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
    f[0] = lo.x; f[1] = lo.y; f[2] = hi.x; f[3] = hi.y;
}

// four floats -> four e4m3 codes (round to nearest even, no saturation)
DEV u32 pack_fp8x4(float a, float b, float c, float d)
{
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
    return (u32)w;
}

// ---------------------------------------------------------------------------
// element types
// ---------------------------------------------------------------------------
template <typename T> struct Elem;

template <> struct Elem<float> {
    static constexpr int ESZ = 4;
    static constexpr int EPV = 4;  // elements per 16-byte vector
    DEV static void unpack(const u32x4 v, float (&f)[4])
    {
        f[0] = as_f(v.x); f[1] = as_f(v.y); f[2] = as_f(v.z); f[3] = as_f(v.w);
    }
    DEV static u32x4 pack(const float (&f)[4])
    {
        u32x4 v = {as_u(f[0]), as_u(f[1]), as_u(f[2]), as_u(f[3])};
        return v;
    }
    DEV static float load(uint64_t base, int64_t idx) { return as_global<const float>(base)[idx]; }
    DEV static void store(uint64_t base, int64_t idx, float v) { as_global<float>(base)[idx] = v; }
    DEV static float rounded(float v) { return v; }  // v as a stored element reads back
    // elements idx and idx + 1 with one access (streaming: neighbouring lanes take neighbouring
    // pairs, so a wavefront covers whole lines)
    DEV static void load2(uint64_t base, int64_t idx, float &a, float &b)
    {
        const u32x2 w = LOAD_STREAM((GLOBAL const u32x2_a4 *)(as_global<const float>(base) + idx));
        a = as_f(w.x);
        b = as_f(w.y);
    }
    DEV static void store2(uint64_t base, int64_t idx, float a, float b)
    {
        const u32x2 w = {as_u(a), as_u(b)};
        STORE_STREAM(w, (GLOBAL u32x2_a4 *)(as_global<float>(base) + idx));
    }
};

template <> struct Elem<bf16_tag> {
    static constexpr int ESZ = 2;
    static constexpr int EPV = 8;
    DEV static void unpack(const u32x4 v, float (&f)[8])
    {
        f[0] = as_f(v.x << 16); f[1] = as_f(v.x & 0xFFFF0000u);
        f[2] = as_f(v.y << 16); f[3] = as_f(v.y & 0xFFFF0000u);
        f[4] = as_f(v.z << 16); f[5] = as_f(v.z & 0xFFFF0000u);
        f[6] = as_f(v.w << 16); f[7] = as_f(v.w & 0xFFFF0000u);
    }
    DEV static u32 pack2(float a, float b)
    {
        const f32x2 p = {a, b};
        const bf16x2 h = __builtin_convertvector(p, bf16x2);  // round to nearest even
        return __builtin_bit_cast(u32, h);
    }
    DEV static u32x4 pack(const float (&f)[8])
    {
        u32x4 v = {pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]), pack2(f[6], f[7])};
        return v;
    }
    DEV static float load(uint64_t base, int64_t idx)
    {
        return as_f((u32)as_global<const uint16_t>(base)[idx] << 16);
    }
    DEV static void store(uint64_t base, int64_t idx, float v)
    {
        as_global<uint16_t>(base)[idx] = (uint16_t)(pack2(v, 0.0f) & 0xFFFFu);
    }
    DEV static float rounded(float v) { return as_f(pack2(v, 0.0f) << 16); }
    DEV static void load2(uint64_t base, int64_t idx, float &a, float &b)
    {
        const u32 w = LOAD_STREAM((GLOBAL const u32_a2 *)(as_global<const uint16_t>(base) + idx));
        a = as_f(w << 16);
        b = as_f(w & 0xFFFF0000u);
    }
    DEV static void store2(uint64_t base, int64_t idx, float a, float b)
    {
        STORE_STREAM(pack2(a, b), (GLOBAL u32_a2 *)(as_global<uint16_t>(base) + idx));
    }
};

template <> struct Elem<f16_tag> {
    static constexpr int ESZ = 2;
    static constexpr int EPV = 8;
    DEV static void unpack2(u32 w, float &a, float &b)
    {
        const f16x2 h = __builtin_bit_cast(f16x2, w);
        a = (float)h.x;
        b = (float)h.y;
    }
    DEV static void unpack(const u32x4 v, float (&f)[8])
    {
        unpack2(v.x, f[0], f[1]); unpack2(v.y, f[2], f[3]);
        unpack2(v.z, f[4], f[5]); unpack2(v.w, f[6], f[7]);
    }
    // The value is first rounded to binary32, then to binary16.  Hide the
    // producer from the compiler: it would otherwise fuse fma + convert into
    // v_fma_mixlo_f16, which rounds once and differs in the last bit.
    DEV static float opaque(float x)
    {
        asm("" : "+v"(x));
        return x;
    }
    DEV static u32 pack2(float a, float b)
    {
        f16x2 h;
        h.x = (_Float16)opaque(a);  // round to nearest even
        h.y = (_Float16)opaque(b);
        return __builtin_bit_cast(u32, h);
    }
    DEV static u32x4 pack(const float (&f)[8])
    {
        u32x4 v = {pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]), pack2(f[6], f[7])};
        return v;
    }
    DEV static float load(uint64_t base, int64_t idx)
    {
        return (float)as_global<const _Float16>(base)[idx];
    }
    DEV static void store(uint64_t base, int64_t idx, float v)
    {
        as_global<_Float16>(base)[idx] = (_Float16)opaque(v);
    }
    DEV static float rounded(float v) { return (float)(_Float16)opaque(v); }
    DEV static void load2(uint64_t base, int64_t idx, float &a, float &b)
    {
        unpack2(LOAD_STREAM((GLOBAL const u32_a2 *)(as_global<const uint16_t>(base) + idx)), a, b);
    }
    DEV static void store2(uint64_t base, int64_t idx, float a, float b)
    {
        STORE_STREAM(pack2(a, b), (GLOBAL u32_a2 *)(as_global<uint16_t>(base) + idx));
    }
};

// The elements in one dword of a tensor: one (fp32) or two.
template <typename T>
DEV void unpack_dword(u32 w, float (&f)[4 / Elem<T>::ESZ])
{
    if constexpr (std::is_same<T, float>::value) f[0] = as_f(w);
    else if constexpr (std::is_same<T, f16_tag>::value) Elem<T>::unpack2(w, f[0], f[1]);
    else {
        f[0] = as_f(w << 16);
        f[1] = as_f(w & 0xFFFF0000u);
    }
}

// ---------------------------------------------------------------------------
// workgroup -> (segment, first row)
// ---------------------------------------------------------------------------
// Consecutive workgroup ids are dealt round-robin to the 8 XCDs, each with its
// own L2.  Workgroup id b is the (b >> 3)-th piece of work of XCD b & 7.
//
// Inline table (at most 16 segments): XCD x takes the x-th contiguous eighth of
// every segment's workgroups and walks the segments in the stage's work order
// (reduce: heaviest workgroups first, so that every XCD sees the same mix of
// row lengths and the last workgroups to finish are light).
// Device table (longer lists): workgroup numbers follow the segments in the
// stage's work order, chunks of consecutive numbers go to the XCDs in turn, and
// a bucket map plus a short binary search lead from the number to the segment.
// Ids past the end of their XCD's work return false.
//
// A list of one tensor needs no round of scalar loads (KOne: its arguments are in registers when the
// wavefront starts), a longer one two or three.  A kernel that is one round of workgroups is that much
// shorter: with the tables of a longer list, with KOne loaded as a structure and with KOne in registers,
// quantize, reduce and dequantize of a bf16 [4096, 4096] for 8 peers 11.5, 6.4, 12.6 / 10.8, 6.0, 11.7 /
// 10.8, 5.9, 11.4 us, of 315 fp32 elements 2.1, 3.2, 2.1 / 1.7, 2.9, 1.6 / 1.4, 2.5, 1.4 us.  (The
// descriptors of up to four tensors loaded in one round and selected in registers gain nothing: 64
// scalar registers and their selection cost what the second round does.)
//
// Indexing by-value kernel arguments with a run-time index would make the compiler copy them to
// private memory; reading the kernel-argument segment through a constant-address-space pointer keeps
// the accesses scalar loads.
#define CONSTANT __attribute__((address_space(4)))

// locate<STAGE>(kernel arguments, call, segment, workgroup of the segment); false: nothing to do.
// KOne as kernel parameters, of which -amdgpu-kernarg-preload-count puts the first 56 bytes into
// scalar registers, and back.
#define TFTQ_ONE_PARAMS                                                                                            \
    const uint64_t w0, const uint64_t w1, const uint64_t w2, const uint64_t w3, const uint64_t w4, const uint64_t w5, \
        const uint64_t w6, const uint64_t w7
#define TFTQ_ONE w0, w1, w2, w3, w4, w5, w6, w7
DEV KOne one_of(TFTQ_ONE_PARAMS)
{
    const uint64_t w[8] = {TFTQ_ONE};
    return __builtin_bit_cast(KOne, w);
}

template <int STAGE>
DEV bool locate(const KOne &a, KCall &p, Seg &s, int &blk)
{
    constexpr bool R = STAGE == ST_R;
    blk = tftq_one_piece(a.nwg, a.natural, blockIdx.x);
    s.ptr = R ? 0 : a.ptr;
    s.slot_off = 0;
    s.row_stride = R ? 0 : a.row_stride;
    s.col_stride = R ? 0 : a.col_stride;
    s.m = a.m;
    s.n = a.n;
    s.slice_rows = a.slice_rows;
    s.row_bytes = ((a.n + 3) & ~3) + 4;
    s.kind[STAGE] = a.kind;
    s.side = a.side;
    s.lg_groups = a.lg_groups;
    p.packed = a.packed;
    p.slot_size = (int64_t)a.slice_rows * s.row_bytes;
    p.ws = a.ws;
    p.rank = R ? a.rank : 0;
    p.div_mode = a.div_mode;
    p.div = R ? a.div : 1.0f;
    p.inv_div = R ? a.inv_div : 1.0f;
    p.post_scale = a.post_scale;
    return blk >= 0;
}

template <int STAGE>
DEV bool locate(const KInline &a, KCall &p, Seg &s, int &blk)
{
    const int x = (int)(blockIdx.x & 7);
    int i = (int)(blockIdx.x >> 3);
    // One round of scalar loads fetches this XCD's three table rows; the position
    // is then found in registers, and only the segment descriptor needs a second round.
    const CONSTANT char *karg = (const CONSTANT char *)__builtin_amdgcn_kernarg_segment_ptr();
    const CONSTANT int32_t *d = (const CONSTANT int32_t *)(karg + offsetof(KInline, dealt)) + x * TFTQ_N_INLINE;
    typedef int32_t Row __attribute__((ext_vector_type(TFTQ_N_INLINE)));  // one 64-byte scalar load
    const Row cum_end = *(const CONSTANT Row *)(d + offsetof(Dealt, cum_end) / 4);
    const Row base = *(const CONSTANT Row *)(d + offsetof(Dealt, base) / 4);
    const Row seg = *(const CONSTANT Row *)(d + offsetof(Dealt, seg) / 4);
    Row cum_end_ = cum_end, base_ = base, seg_ = seg;
    // all scalar loads of this round, and the common parameters, are issued before the first wait
    int natural = a.natural;
    asm volatile("" : "+s"(cum_end_), "+s"(base_), "+s"(seg_), "+s"(natural)
                 : "s"(a.call.packed), "s"(a.call.slot_size), "s"(a.call.ws), "s"(a.call.rank));
    p = a.call;
    if (natural) i = (int)blockIdx.x;  // all eight rows of the table describe the whole work
    int b = base_[0], sg = seg_[0];
#pragma unroll
    for (int j = 1; j < TFTQ_N_INLINE; j++) {
        const bool past = i >= cum_end_[j - 1];  // cum_end is non-decreasing: the last hit wins
        b = past ? base_[j] : b;
        sg = past ? seg_[j] : sg;
    }
    if (sg < 0 || i >= cum_end_[TFTQ_N_INLINE - 1]) return false;
    const CONSTANT u32x4 *src = (const CONSTANT u32x4 *)(karg + offsetof(KInline, s) + (uint64_t)(u32)sg * sizeof(Seg));
    const u32x4 v[4] = {src[0], src[1], src[2], src[3]};
    __builtin_memcpy(&s, v, sizeof(Seg));
    blk = b + i - s.wg_begin[STAGE];
    return true;
}

template <int STAGE>
DEV bool locate(const KTable &a, KCall &p, Seg &s, int &blk)
{
    const int x = (int)(blockIdx.x & 7), i = (int)(blockIdx.x >> 3);
    // everything the first steps need from the kernel arguments in one round of scalar loads
    asm volatile("" ::"s"(a.table), "s"(a.ptrs), "s"(a.map_off), "s"(a.sorted_off), "s"(a.map_shift), "s"(a.chunk_shift),
                 "s"(a.nwg), "s"(a.pieces), "s"(a.call.packed), "s"(a.call.slot_size), "s"(a.call.ws), "s"(a.call.rank));
    p = a.call;
    // chunks of 2^chunk_shift consecutive workgroups go to the XCDs in turn
    const int cs = a.chunk_shift;
    int vb = ((((i >> cs) << 3) + x) << cs) + (i & ((1 << cs) - 1));
    if (vb >= a.nwg) return false;
    if (STAGE == ST_R && a.pieces) {  // this wavefront's quarter of the workgroup (tftq_reduce_pieces)
        vb = 4 * vb + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        if (vb >= a.pieces) return false;
    }
    const uint64_t tab = (uint64_t)a.table;
    typedef int32_t MapPair __attribute__((ext_vector_type(4), aligned(8)));
    const MapPair m = *(const CONSTANT MapPair *)(tab + (uint64_t)a.map_off +
                                                  (uint64_t)(vb >> a.map_shift) * sizeof(MapEnt));
    int lo = m.x, sg = m.y, hi = m.z;
    if (lo != hi) {  // last position whose first workgroup is <= vb
        const CONSTANT SortEnt *sorted = (const CONSTANT SortEnt *)(tab + (uint64_t)a.sorted_off);
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (sorted[mid].begin <= vb) lo = mid; else hi = mid - 1;
        }
        sg = sorted[lo].seg;
    }
    const CONSTANT u32x4 *src = (const CONSTANT u32x4 *)(tab + (uint64_t)sg * sizeof(Seg));
    const u32x4 v[4] = {src[0], src[1], src[2], src[3]};
    // the table holds no addresses: the tensor's comes from the call's pointer array
    uint64_t tptr = 0;
    if (STAGE != ST_R) tptr = *(const CONSTANT uint64_t *)((uint64_t)a.ptrs + (uint64_t)sg * 8u);
    __builtin_memcpy(&s, v, sizeof(Seg));
    s.ptr = tptr;
    blk = vb - s.wg_begin[STAGE];
    return true;
}

DEV int64_t row_addr(const Seg &s, int64_t slot_size, int row)
{
    const int slot = row / s.slice_rows;
    const int j = row - slot * s.slice_rows;
    return (int64_t)slot * slot_size + s.slot_off + (int64_t)j * s.row_bytes;
}

// Short contiguous rows of whole 16-byte vectors (K_VECS; the shape is
// tftq_small_shape): 1 to 32 lanes per row, and every lane works on several rows
// so that it has 8 loads in flight.  Row slot r of team t is row
// row0 + r * teams + t: for a given r the teams of a wavefront read
// consecutive rows, i.e. consecutive memory.
struct SmallShape {
    int lt, c, team, teams, t, l;
};
DEV SmallShape small_shape(int nvec, int tid, int stage)
{
    SmallShape h;
    tftq_small_shape(nvec, &h.lt, &h.c, stage);
    h.team = 1 << h.lt;
    h.teams = TFTQ_WG >> h.lt;
    h.t = tid >> h.lt;
    h.l = tid & (h.team - 1);
    return h;
}

// row -> byte offset of the packed row, with the slot found by one multiply
// (inv = 1.0f / slice_rows; the estimate is off by at most one)
DEV int64_t row_addr_fast(const Seg &s, int64_t slot_size, int row, float inv)
{
    int slot = (int)((float)row * inv);
    int j = row - slot * s.slice_rows;
    if (j < 0) { --slot; j += s.slice_rows; }
    if (j >= s.slice_rows) { ++slot; j -= s.slice_rows; }
    return (int64_t)slot * slot_size + s.slot_off + (int64_t)j * s.row_bytes;
}

// ---------------------------------------------------------------------------
// packed rows through LDS
// ---------------------------------------------------------------------------
// Staging of a workgroup's packed rows in LDS.  The rows that one workgroup quantizes are
// neighbours in the packed buffer, so together they are one span of bytes; packed rows
// start anywhere (4 + n bytes each), which makes direct stores cover parts of 128-byte
// lines with every instruction.  The workgroup instead assembles the span in LDS, at the
// offset that the span has inside its first 128-byte line, and then copies it out with
// streaming 16-byte stores whose wavefronts each cover eight whole lines; only the first
// and the last 16 bytes of the span can be partial and go out as halfwords.
#define LDS_AS __attribute__((address_space(3)))

template <int LANES = TFTQ_WG>
DEV void copy_out_span(const uint8_t *stage, uint8_t *g0, int len, int tid)
{
    const int mis = (int)((uintptr_t)g0 & 127u);
    GLOBAL uint8_t *line0 = as_global<uint8_t>(g0 - mis);  // stage[x] belongs at line0[x]
    const int end = mis + len;
    const int nchunks = (end + 15) >> 4;
#pragma nounroll
    for (int c = tid; c < nchunks; c += LANES) {
        const int lo = 16 * c;
        const u32x4 v = *(const LDS_AS u32x4 *)(const LDS_AS uint8_t *)(stage + lo);
        if (lo >= mis && lo + 16 <= end) {
            STORE_STREAM(v, (GLOBAL u32x4 *)(line0 + lo));
        } else {  // the span's first or last 16 bytes: halfwords (a span starts and ends at even bytes)
            const u32 w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int d = 0; d < 8; d++)
                if (lo + 2 * d >= mis && lo + 2 * d < end)
                    *(GLOBAL uint16_t *)(line0 + lo + 2 * d) = (uint16_t)(w[d >> 1] >> (16 * (d & 1)));
        }
    }
}

// ---------------------------------------------------------------------------
// host side: kernel arguments of a launch
// ---------------------------------------------------------------------------
struct KArgs {
    enum { ONE, INLINE, TABLE } where;
    unsigned grid;
    union {
        KOne one;
        KInline inl;
        KTable table;
    };
    KArgs() {}
};

// Makes `device` current for the lifetime of the object and restores the caller's device
// afterwards; device < 0 leaves the current device alone.
struct DeviceScope {
    int prev = -1;
    bool switched = false;
    hipError_t err = hipSuccess;
    explicit DeviceScope(int device)
    {
        if (device < 0) return;
        err = hipGetDevice(&prev);
        if (err == hipSuccess && prev != device) {
            err = hipSetDevice(device);
            switched = err == hipSuccess;
        }
    }
    ~DeviceScope()
    {
        if (switched) (void)hipSetDevice(prev);
    }
    DeviceScope(const DeviceScope &) = delete;
    DeviceScope &operator=(const DeviceScope &) = delete;
};

// Copies `bytes` bytes (a multiple of 8) from host memory to 8-byte aligned device memory
// with small kernels on `st` that carry the data in their arguments: the source is read
// before the function returns, nothing is allocated or synchronised, and a stream capture
// records the data itself.  Defined in tftq_runtime.hip.
__attribute__((visibility("hidden"))) int tftq_put_bytes(void *dst_device, const void *src_host, size_t bytes,
                                                         hipStream_t st);

// Looks up, for the current device, the address of the fixed array that tftq_reduce_static
// keeps its table in.  Defined in tftq_reduce.hip.
__attribute__((visibility("hidden"))) int tftq_static_table_setup(void);

// One kernel launch with the launch's own error (not whatever an earlier call left behind).
template <typename K, typename A>
static inline int launch_kernel(K kernel, const KArgs &ka, const A &arg, unsigned lds_bytes, hipStream_t st, int threads = TFTQ_WG)
{
    void *args[8];
    const bool one = std::is_same<A, KOne>::value;  // eight words
    for (int i = 0; i < (one ? 8 : 1); i++) args[i] = (char *)&arg + 8 * i;
    return (int)hipLaunchKernel((const void *)kernel, dim3(ka.grid), dim3(threads), args, lds_bytes, st);
}

// f(the arguments) with the type of the list's length.
template <typename F>
static inline int with_args(const KArgs &ka, F f)
{
    switch (ka.where) {
    case KArgs::ONE: return f(ka.one);
    case KArgs::INLINE: return f(ka.inl);
    default: return f(ka.table);
    }
}

// What a call of a stage must bring along: tensors, a host array of the tensors' device addresses
// (null in reduce); table and pointers, the caller's device buffers of a long list.
static inline int check_call(const tftq_plan *plan, int stage, const void *const *tensors, const void *table,
                             const void *pointers, const void *packed, int64_t packed_bytes)
{
    if (!plan) return TFTQ_E_ARG;
    if (packed_bytes != plan->output_size) return TFTQ_E_SIZE;
    // a list of empty tensors has an empty packed buffer, whose address may be null
    if (!packed && plan->output_size != 0) return TFTQ_E_ARG;
    if (((uintptr_t)packed & 3) != 0) return TFTQ_E_ARG;
    const bool needs_tensors = stage != ST_R && plan->nwg[stage] > 0;
    auto missing = [&](int i) { return !tensors[i] && plan->segs[(size_t)i].m > 0 && plan->segs[(size_t)i].n > 0; };
    if (plan->nseg <= TFTQ_N_INLINE) {
        if (needs_tensors && !tensors) return TFTQ_E_ARG;
        if (stage == ST_R) return 0;
    } else {
        if (plan->nwg[stage] == 0) return 0;
        if (!table || ((uintptr_t)table & 255) != 0) return TFTQ_E_NOTABLE;
        if (!needs_tensors) return 0;
        if (!pointers || ((uintptr_t)pointers & 7) != 0) return TFTQ_E_NOTABLE;
        if (!tensors) return 0;
    }
    for (int i = 0; i < plan->nseg; i++)
        if (tensors ? missing(i) : plan->segs[(size_t)i].m > 0 && plan->segs[(size_t)i].n > 0) return TFTQ_E_ARG;
    return 0;
}

// Writes the addresses of a long list's tensors, where the call has them, to `pointers` on `st`.
static inline int put_addresses(const tftq_plan *plan, const void *const *tensors, void *pointers, hipStream_t st)
{
    return tensors && plan->nseg > TFTQ_N_INLINE ? tftq_put_bytes(pointers, tensors, (size_t)plan->nseg * 8, st) : 0;
}

constexpr KCall PLAIN_CALL = {nullptr, 0, 0, 0, 0, 1.0f, 1.0f, 1.0f};

// The kernel arguments of a launch.  what: all but packed, slot_size and ws, which the plan knows.
static inline void fill_args(const tftq_plan *plan, int stage, const void *const *tensors, const void *table,
                             const void *pointers, void *packed, const KCall &what, KArgs *ka)
{
    const int field = stage == ST_QC ? (int)ST_Q : stage;
    const bool natural = plan->nseg <= TFTQ_N_INLINE && plan->natural[stage];
    auto address = [&](int i) { return stage == ST_R || !tensors ? (uint64_t)0 : (uint64_t)(uintptr_t)tensors[i]; };
    ka->grid = 8u * (unsigned)(plan->nseg <= TFTQ_N_INLINE ? plan->dealt_per_xcd[stage] : plan->index[stage].per_xcd);
    if (plan->nseg == 1) {
        const Seg &s = plan->segs[0];
        KOne &a = ka->one;
        ka->where = KArgs::ONE;
        a.packed = (uint8_t *)packed;
        if (stage == ST_R) {
            a.rank = what.rank;
            a.div = what.div;
            a.inv_div = what.inv_div;
        } else {
            a.ptr = address(0);
            a.row_stride = s.row_stride;
            a.col_stride = s.col_stride;
        }
        a.m = s.m;
        a.n = s.n;
        a.slice_rows = s.slice_rows;
        a.ws = plan->ws;
        a.nwg = plan->nwg[stage];
        a.kind = s.kind[field];
        a.side = s.side;
        a.lg_groups = s.lg_groups;
        a.natural = natural;
        a.div_mode = (uint8_t)what.div_mode;
        a.post_scale = what.post_scale;
        return;
    }
    KCall call = what;
    call.packed = (uint8_t *)packed;
    call.slot_size = plan->slot_size;
    call.ws = plan->ws;
    if (plan->nseg <= TFTQ_N_INLINE) {
        KInline &a = ka->inl;
        ka->where = KArgs::INLINE;
        a.call = call;
        a.natural = natural;
        a.dealt = plan->dealt[stage];
        for (int i = 0; i < plan->nseg; i++) {
            a.s[i] = plan->segs[(size_t)i];
            a.s[i].ptr = address(i);
        }
    } else {
        const TableIndex &index = plan->index[stage];
        KTable &a = ka->table;
        ka->where = KArgs::TABLE;
        a.call = call;
        a.table = (const Seg *)table;
        a.ptrs = stage == ST_R ? nullptr : (const uint64_t *)pointers;
        a.nwg = plan->nwg[stage];
        a.pieces = index.pieces;
        a.map_shift = index.shift;
        a.chunk_shift = index.chunk_shift;
        a.sorted_off = index.sorted_off;
        a.map_off = index.map_off;
    }
}
