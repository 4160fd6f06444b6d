// FLAT in slices of K: one pass over the stored entries per 128 bytes of the rows.
//
// What bounds the gather kernels on rows of several lines is the interface between the L2s and the
// last-level cache: a launch touches all of B at any moment, B does not fit the 4 MB L2 of an XCD, and
// every gathered line crosses that interface (7.3 TB/s measured; 705 k entries of 4 000-byte rows:
// 40 M lines, 700 us).  Here the work is ordered by slice first: workgroup (s, e) takes slice s -- one
// line of every B row -- of a range of entries, workgroups go to the XCDs in that order (xcd_remap), so
// an XCD works on one slice of B at a time, N * 128 bytes, and the lines are found in its L2 (the
// same launch: 7 M lines from the last-level cache, 200 us, now bound by the CU's vector memory path:
// 28 cycles per gathered 1 KiB).  The partial products of a slice, one float per entry, go to a
// workspace; k_slice_sum adds them up (in k order, so the result does not depend on the schedule) and
// multiplies by S: 8 bytes per entry and slice, against the 128 bytes of its B line.
//
// Slices are lines of memory, not of the row: a B row that does not start on a line (its length is no
// multiple of 128 bytes) has its window moved down to the line, so that every gather is one line.  The
// A row of an entry must then be read at the same, per-entry position: the A rows of a wavefront's 256
// entries are few (entries come row by row), so their 256 bytes around the slice go to LDS once and are
// read from there at any position.  Entries in no order, or rows of one or two entries, span more than
// SLICE_ROWS rows: those wavefronts gather A like B.
//
// Lane layout: 8 neighbouring lanes share one entry, group g of lanes takes entries 8g .. 8g+7 of a
// chunk of 64, one per step; step t's total stays in lane 8g+t, which is the lane of that entry.
#pragma once
#include "kernels_gather.h"

namespace sddmm {

constexpr int SLICE_BYTES = 128;                   // one line of B per entry and pass
constexpr int SLICE_LPN = 8;                       // lanes per entry
constexpr int SLICE_ROWS = 24;                     // distinct A rows of a wavefront's entries that are staged in LDS
constexpr int SLICE_CHUNKS = 4;                    // chunks of 64 entries per wavefront (2: 216 us, 8: 212, 16: 270 against 219)
constexpr int SLICE_ENTRIES = SLICE_CHUNKS * WAVE;

// MISALIGNED: some B row does not start on a line; UNALIGNED: rows are only 4-byte aligned (K % 4 in fp32)
template <class U, bool MISALIGNED, bool UNALIGNED, bool WIDE>
__global__ __launch_bounds__(BLOCK, 4) void k_slice_dots(int64_t nblocks, int64_t blocks_per_slice, int64_t nnz,
    const int32_t *__restrict__ rowidx, const int32_t *__restrict__ col, const void *__restrict__ A,
    const void *__restrict__ B, int row_bytes, float *__restrict__ part, int64_t stride) {
    static_assert(MISALIGNED || !UNALIGNED, "rows of no whole number of units are misaligned");
    using T = typename U::T;
    using O = typename Off<WIDE>::T;
    constexpr int LPN = SLICE_LPN, C = SLICE_CHUNKS;
    // a staged A row: the slice's 128 bytes and, where windows move down, the 128 before them; 16 more in
    // front where the last 16 bytes of a row can begin before those
    constexpr int FRONT = UNALIGNED ? 16 : 0;
    constexpr int WINDOW = MISALIGNED ? 2 * SLICE_BYTES : SLICE_BYTES;
    constexpr int PITCH = FRONT + WINDOW;
    constexpr int LPR = WINDOW / 16, RPL = WAVE / LPR;      // lanes per staged row, rows per staging load
    __shared__ __attribute__((aligned(16))) uint32_t b_all[WAVES_PER_BLOCK][SLICE_ENTRIES], a_all[WAVES_PER_BLOCK][SLICE_ENTRIES];
    __shared__ __attribute__((aligned(16))) char rows_all[WAVES_PER_BLOCK][SLICE_ROWS * PITCH];
    __shared__ uint32_t list_all[WAVES_PER_BLOCK][SLICE_ROWS];
    const int64_t blk = xcd_remap(blockIdx.x, nblocks);
    if (blk < 0) return;
    const int64_t slice = blk / blocks_per_slice;
    const int lane = lane_id(), wv = wave_in_block();
    const int64_t base = ((blk - slice * blocks_per_slice) * WAVES_PER_BLOCK + wv) * SLICE_ENTRIES;
    if (base >= nnz) return;                                // (no workgroup barrier below)
    const int s = (int)slice;
    const int g = lane / LPN, j = lane & (LPN - 1);
    uint32_t *b_at = b_all[wv], *a_at = a_all[wv], *row_list = list_all[wv];
    char *rows = rows_all[wv];
    uint32_t *mis_at = (uint32_t *)rows;                    // misalignments of entries whose A rows are not staged
    static_assert(SLICE_ENTRIES * 4 <= SLICE_ROWS * PITCH, "the misalignments fit the unused row buffer");
    const int64_t last = nnz - 1;
    const uint32_t b_low = (uint32_t)(uintptr_t)B;
    auto row_off = [&](uint32_t v) { return (O)v * (O)(uint32_t)row_bytes; };
    // bytes from the line a B row starts in to its start
    auto misalignment = [&](O off) { return MISALIGNED ? (b_low + (uint32_t)off) & (SLICE_BYTES - 1) : 0u; };
    // b_at: line of the entry's B row as a byte offset (WIDE: the row).  a_at: the entry's row among the
    // staged ones and the misalignment of its B row (not staged: the row, and mis_at).
    int distinct = 0;
    {
        int r[C], rank[C];
        uint32_t cc[C], mis[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int64_t n = base + c * WAVE + lane;
            const int64_t at = n < last ? n : last;         // entries past the end repeat the last one, unstored
            r[c] = rowidx[at];
            cc[c] = (uint32_t)col[at];
        }
        int carry = -1;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            // row of the entry before: lane - 1 (wave_shr:1), for lane 0 the last entry of the chunk before
            const int before = __builtin_amdgcn_update_dpp(carry, r[c], 0x138, 0xF, 0xF, false);
            carry = __builtin_amdgcn_readlane(r[c], WAVE - 1);
            const bool starts = r[c] != before;
            const unsigned long long m = __ballot(starts);
            rank[c] = distinct + __popcll(m & (~0ull >> (WAVE - 1 - lane))) - 1;
            distinct += __popcll(m);
            if (starts && rank[c] < SLICE_ROWS) row_list[rank[c]] = (uint32_t)r[c];
            const O off = row_off(cc[c]);
            mis[c] = misalignment(off);
            b_at[c * WAVE + lane] = WIDE ? cc[c] : (uint32_t)off - mis[c];
        }
        const bool staged = distinct <= SLICE_ROWS;         // wave-uniform
#pragma unroll
        for (int c = 0; c < C; ++c) {
            a_at[c * WAVE + lane] = staged ? (uint32_t)(rank[c] * PITCH) * SLICE_BYTES + mis[c] : (uint32_t)r[c];
            if (MISALIGNED && !staged) mis_at[c * WAVE + lane] = mis[c];
        }
    }
    wave_lds_order();
    struct Eight { uint32_t x[LPN]; };
    auto eight = [&](const uint32_t *p) {                   // the steps of this lane's group
        const uint4 lo = *reinterpret_cast<const uint4 *>(p), hi = *reinterpret_cast<const uint4 *>(p + 4);
        return Eight{{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w}};
    };
    auto load16 = [&](const void *p, O off) {
        const char *at = reinterpret_cast<const char *>(p) + off;
        if constexpr (UNALIGNED) return __builtin_bit_cast(T, *reinterpret_cast<const I4u *>(at));
        else return *reinterpret_cast<const T *>(at);
    };
    const int here = s * SLICE_BYTES + j * 16;              // byte inside a line-aligned row that this lane takes
    const int top = row_bytes - 16;
    auto inside = [&](int x) { return x < 0 ? 0 : x < top ? x : top; };
    // every lane of every entry inside its row?  (wave-uniform; else positions are clamped and masked)
    const bool inner = !MISALIGNED || (s > 0 && s < row_bytes / SLICE_BYTES);

    auto walk = [&](auto nr_tag) {
        constexpr int NR = decltype(nr_tag)::value;         // loads that stage the A rows; 0: A gathered per entry
        const int first = MISALIGNED ? (s - 1) * SLICE_BYTES : s * SLICE_BYTES;      // byte of a row that is staged first
        const int xa = inside(first + (lane & (LPR - 1)) * 16);
        T ar[NR > 0 ? NR : 1];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int rr = i * RPL + lane / LPR;
            ar[i] = load16(A, row_off(row_list[rr < distinct ? rr : 0]) + (O)xa);
        }
        auto mis_of = [&](const Eight &ea, int c) {         // misalignments of the group's entries of chunk c
            Eight m;
            if constexpr (NR == 0) m = MISALIGNED ? eight(mis_at + c * WAVE + g * LPN) : Eight{};
            else for (int t = 0; t < LPN; ++t) m.x[t] = ea.x[t] & (SLICE_BYTES - 1);
            return m;
        };
        auto load_b = [&](int c, T (&b)[LPN]) {
            const Eight e = eight(b_at + c * WAVE + g * LPN);
            if (inner) {
#pragma unroll
                for (int t = 0; t < LPN; ++t) {
                    O off = (O)e.x[t];
                    if constexpr (WIDE) { off = row_off(e.x[t]); off -= misalignment(off); }
                    b[t] = load_at<T, O>(B, off + (O)(uint32_t)here);
                }
            } else {
                const Eight m = mis_of(eight(a_at + c * WAVE + g * LPN), c);
#pragma unroll
                for (int t = 0; t < LPN; ++t) {
                    const O off = WIDE ? row_off(e.x[t]) : (O)(e.x[t] + m.x[t]);
                    b[t] = load16(B, off + (O)(uint32_t)inside(here - (int)m.x[t]));
                }
            }
        };
        T bf[2][LPN];
        load_b(0, bf[0]);
        if constexpr (NR > 0) {
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                char *dst = rows + (i * RPL + lane / LPR) * PITCH + FRONT + (xa - first);
                if constexpr (UNALIGNED) *reinterpret_cast<I4u *>(dst) = __builtin_bit_cast(I4u, ar[i]);
                else *reinterpret_cast<T *>(dst) = ar[i];
            }
            wave_lds_order();
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            T (&cur)[LPN] = bf[c & 1];
            const Eight ea = eight(a_at + c * WAVE + g * LPN);
            const Eight m = mis_of(ea, c);
            T af[NR > 0 ? 1 : LPN];
            if constexpr (NR == 0) {
#pragma unroll
                for (int t = 0; t < LPN; ++t) af[t] = load16(A, row_off(ea.x[t]) + (O)(uint32_t)inside(here - (int)m.x[t]));
            }
            if (c + 1 < C) load_b(c + 1, bf[(c + 1) & 1]);
            auto a_unit = [&](int t, int x) {                // 16 bytes from byte x of entry t's A row
                if constexpr (NR == 0) return af[t];
                else {
                    const char *src = rows + (ea.x[t] / SLICE_BYTES + (uint32_t)(FRONT - first + x));
                    if constexpr (UNALIGNED) return __builtin_bit_cast(T, *reinterpret_cast<const I4u *>(src));
                    else return *reinterpret_cast<const T *>(src);
                }
            };
            float out = 0.f;
            auto keep = [&](int t, float p) {
                p = group_sum<LPN>(p);
                out = j == t ? p : out;
            };
            if (inner) {
#pragma unroll
                for (int t = 0; t < LPN; ++t) keep(t, U::dot(a_unit(t, here - (int)m.x[t]), cur[t], 0.f));
            } else {
#pragma unroll
                for (int t = 0; t < LPN; ++t) {
                    // both operands were read at the clamped position: what lies outside the lane's own 16
                    // bytes belongs to another lane, or to no one, and must not enter even as 0 * inf
                    const int x = here - (int)m.x[t], xc = inside(x);
                    T a = a_unit(t, xc), b = cur[t];
                    if constexpr (UNALIGNED) {
                        float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const bool on = (unsigned int)(xc + 4 * e - x) < 16u;
                            av[e] = on ? av[e] : 0.f;
                            bv[e] = on ? bv[e] : 0.f;
                        }
                        a = make_float4(av[0], av[1], av[2], av[3]);
                        b = make_float4(bv[0], bv[1], bv[2], bv[3]);
                    }
                    const float p = U::dot(a, b, 0.f);
                    keep(t, UNALIGNED || x == xc ? p : 0.f);
                }
            }
            const int64_t n = base + c * WAVE + lane;
            if (n < nnz) part[slice * stride + n] = out;
        }
    };
    if (distinct <= 2 * RPL) walk(std::integral_constant<int, 2>{});
    else if (distinct <= SLICE_ROWS) walk(std::integral_constant<int, SLICE_ROWS / RPL>{});
    else walk(std::integral_constant<int, 0>{});
}

// P = S o (sum of the slices' partial products), four entries per thread; the sum alone without sval
static __global__ __launch_bounds__(BLOCK) void k_slice_sum(const float *__restrict__ part, int slices, int64_t stride,
                                                            const float *__restrict__ sval, float *__restrict__ P,
                                                            int64_t nnz) {
    const int64_t n = ((int64_t)blockIdx.x * BLOCK + threadIdx.x) * 4;
    if (n >= nnz) return;
    f32x4_t sum = *reinterpret_cast<const f32x4_t *>(part + n);
#pragma unroll 8
    for (int s = 1; s < slices; ++s) sum += *reinterpret_cast<const f32x4_t *>(part + s * stride + n);
    if (n + 4 <= nnz) {
        const F4u v = sval ? *reinterpret_cast<const F4u *>(sval + n) : F4u{1.f, 1.f, 1.f, 1.f};
        *reinterpret_cast<F4u *>(P + n) = F4u{sum[0] * v.x, sum[1] * v.y, sum[2] * v.z, sum[3] * v.w};
    } else {
        for (int i = 0; n + i < nnz; ++i) P[n + i] = sum[i] * (sval ? sval[n + i] : 1.f);
    }
}

// Entries that came in no order (a COO edge list) are computed in the plan's order: sorted by row and, inside a
// row, by column block, so that an A row is found in the L1 by the entries after its first and the long rows can be
// cut into column blocks.  The dot products are written in that order and this kernel brings them back:
// entry n was the place[n]-th.  1.2 M edges in no order, K = 75: 82.8 us in their own order, 52.8 us sorted; 72.9 us
// when the kernel that computes them writes P and reads S at scattered places itself (partial lines from eight L2s).
static __global__ __launch_bounds__(BLOCK) void k_unsort(const float *__restrict__ dots, const int32_t *__restrict__ place,
                                                         const float *__restrict__ sval, float *__restrict__ P, int64_t nnz) {
    const int64_t n = ((int64_t)blockIdx.x * BLOCK + threadIdx.x) * 4;
    if (n >= nnz) return;
    if (n + 4 <= nnz) {
        const I4u q = *reinterpret_cast<const I4u *>(place + n);
        const F4u v = *reinterpret_cast<const F4u *>(sval + n);
        *reinterpret_cast<F4u *>(P + n) = F4u{dots[q.x] * v.x, dots[q.y] * v.y, dots[q.z] * v.z, dots[q.w] * v.w};
    } else {
        for (int64_t i = n; i < nnz; ++i) P[i] = dots[place[i]] * sval[i];
    }
}

}  // namespace sddmm
