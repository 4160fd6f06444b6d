// SDDMM followed by SpMM over the same pattern ("FusedMM"):
//
//     P[i,j] = S[i,j] * <A[i,:], B[j,:]>          (what the SDDMM kernels compute)
//     O[i,:] = sum over stored (i,j) of P[i,j] * B[j,:]
//
// The step that consumes an SDDMM result in the applications the reference names
// (attention-like updates in graph learning); the reference itself stops at P.
// The gathered B row of an entry is used twice while it sits in registers, so the
// second product costs no memory traffic beyond the M x K output.  A and B may be fp32,
// bf16 or fp16 (16-byte units of 4 or 8 elements); P and O are fp32.
//
// k_fusedmm: one wavefront per work item = entries [start,end) of one row (rows longer
// than fused_row_max (16 or 64) entries; shorter ones go to k_fusedmm_rows), in the lane layout
// of the gather kernels: groups of LPN lanes, lane j of a group holds units
// j, j+LPN, ... of the A row, of the entry's B row and of the group's partial output
// row.  After the last entry the partial rows of the 64/LPN groups are added with
// lane permutes; group 0 writes the output row, or, when the row was cut into several
// items, the partial row of its piece.  The kernel of the short rows, launched after it,
// adds the pieces of a row in order (add_pieces; k_add_cut_rows where they are many): O is the same in every run.
#pragma once
#include "kernels_gather.h"

namespace sddmm {

// The output row of a row that k_fusedmm cut into n pieces, by the whole wavefront: lane group g adds pieces g, g + G,
// .. and the groups are added with lane permutes, the same order in every run.  Until then the row of O holds the place of
// its first piece.
template <class L>
__device__ __forceinline__ void add_pieces(const float *__restrict__ parts, float *__restrict__ O, int KU, int64_t row,
                                           int n, int lane) {
    using U = typename L::U;
    constexpr int E = U::ELEMS, LPN = L::LPN, UPL = L::UPL, G = WAVE / LPN;
    using C = Chunk<U, L::LPN, L::UPL, L::FULLK, false, L::WIDE>;
    const int g = lane / LPN, j = lane & (LPN - 1);
    const int64_t K = (int64_t)KU * E;
    float *orow = O + row * K;
    const float *part = parts + (int64_t)__float_as_int(*orow) * K;
    float acc[UPL][E];
#pragma unroll
    for (int i = 0; i < UPL; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) acc[i][e] = 0.f;
#pragma unroll 4
    for (int p = g; p < n; p += G) {
#pragma unroll
        for (int i = 0; i < UPL; ++i) {
            const int u = C::unit_on(j, i, KU) ? j + i * LPN : 0;      // (a lane without a unit adds one it does not write)
#pragma unroll
            for (int e = 0; e < E; e += 4) {
                const float4 v = *reinterpret_cast<const float4 *>(part + p * K + E * u + e);
                acc[i][e] += v.x; acc[i][e + 1] += v.y; acc[i][e + 2] += v.z; acc[i][e + 3] += v.w;
            }
        }
    }
#pragma unroll
    for (int off = LPN; off < WAVE; off <<= 1) {
#pragma unroll
        for (int i = 0; i < UPL; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) acc[i][e] += __shfl_xor(acc[i][e], off, WAVE);
    }
    if (g == 0) {
#pragma unroll
        for (int i = 0; i < UPL; ++i) {
            const int u = j + i * LPN;
            if (!C::unit_on(j, i, KU)) continue;
#pragma unroll
            for (int e = 0; e < E; e += 4)
                *reinterpret_cast<float4 *>(orow + E * u + e) =
                    make_float4(acc[i][e], acc[i][e + 1], acc[i][e + 2], acc[i][e + 3]);
        }
    }
}

// the cut rows among those of a wavefront, one after the other (cut: the lane's row was cut, of `len` entries)
template <class L>
__device__ __forceinline__ void add_cut_rows(const float *__restrict__ parts, float *__restrict__ O, int KU, bool cut,
                                             int64_t row, int len, int seg, int lane) {
    unsigned long long todo = __ballot(cut);
    while (todo) {                                    // wave-uniform
        const int src = __ffsll((long long)todo) - 1;
        todo &= todo - 1;
        const int n = (int)(((unsigned int)__shfl(len, src, WAVE) + (unsigned int)seg - 1u) / (unsigned int)seg);
        add_pieces<L>(parts, O, KU, (int64_t)shfl_off<uint64_t>((uint64_t)row, src), n, lane);
    }
}

// The output rows of the cut rows, a workgroup per row: where one wavefront of the kernel of the short rows would add more
// than FUSED_APART_PIECES pieces, of one very long row or of neighbouring long rows (a graph whose rows are sorted by
// length), and the launch would wait for it: 10 .. 20 ns a piece.  That costs a launch, 3 .. 4 us.  There / here: 1 M rows,
// the first 64 of 50 000 entries, K = 32 478 / 223 us; one row of 2.6 M entries K = 64 253 / 171, K = 256 3 468 / 650; 2.6 M
// rows of a graph sorted by length 1 031 / 984; at the line, one row of 300 000 entries 74.9 / 74.5; below it, 200 000
// sorted rows K = 64 fp16 79.7 / 83.7.
// Thread t takes component group t mod Q, Q the power of two that holds a row, and pieces t/Q, t/Q + threads/Q, ..; the
// sums are added in halves: the same order in every run.
static __global__ __launch_bounds__(FUSED_APART_BLOCK) void k_add_cut_rows(const float *__restrict__ parts, float *__restrict__ O,
                                                                       int K, int seg, const int32_t *__restrict__ rowptr,
                                                                       const int32_t *__restrict__ cut_rows) {
    __shared__ float4 sum[FUSED_APART_BLOCK];
    const int64_t row = cut_rows[blockIdx.x];
    const int quads = K / 4, t = (int)threadIdx.x, threads = (int)blockDim.x;      // (K is a multiple of 4, at most 256)
    int q = 1;
    while (q < quads) q *= 2;
    const int n = (int)(((unsigned int)(rowptr[row + 1] - rowptr[row]) + (unsigned int)seg - 1u) / (unsigned int)seg);
    float4 *orow = reinterpret_cast<float4 *>(O + row * K);
    const float4 *part = reinterpret_cast<const float4 *>(parts + (int64_t)__float_as_int(O[row * K]) * K);
    const int u = t & (q - 1);
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    if (u < quads) {
#pragma unroll 4
        for (int p = t / q; p < n; p += threads / q) {
            const float4 v = part[(int64_t)p * quads + u];
            acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w;
        }
    }
    sum[t] = acc;
    for (int half = threads / 2; half >= q; half /= 2) {
        __syncthreads();
        if (t < half) {
            const float4 v = sum[t + half];
            acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w;
            sum[t] = acc;
        }
    }
    if (t < quads) orow[t] = acc;                     // (every thread has read the place in it before the first barrier)
}

// STEPS: one step after the other, and no more of them than the item has, instead of whole batches of steps (the sums are
// the same bit for bit).  The batches hold the values of several steps and both products in registers (a lane with two fp32
// units 82 instead of 53, with four bf16 units 170 instead of 127): a wavefront is faster and the chip holds fewer of them.
// What that gives and costs (steps / batches): near-dense rows, fewer of them than there are places, K = 128 fp16 75 / 68
// us; dense tiles K = 256 fp16 194 / 151; 3 000 rows of 300 .. 700 entries K = 64 50 / 38; graphs of 50 000 rows K = 64
// 43 / 37.7; 36 000 banded rows that share their columns with their neighbours K = 256 fp16 379 / 310; but 20 000 rows of
// 390 random columns out of 40 000, where the wavefronts in flight walk B together from one end to the other, K = 64
// 120 / 186, K = 192 fp16 246 / 287, and 30 000 rows of 65 .. 127 entries K = 128 bf16 92 / 102 (fused_in_steps: the rule).
template <class L, bool STEPS>
__global__ __launch_bounds__(BLOCK) void k_fusedmm(int64_t nblocks, int64_t n_items, const RowItem *__restrict__ items,
    const int32_t *__restrict__ col, const float *__restrict__ sval, const void *__restrict__ A, const void *__restrict__ B,
    int KU, const int32_t *__restrict__ rowptr, float *__restrict__ P, float *__restrict__ O, float *__restrict__ parts) {
    using U = typename L::U;
    using T = typename U::T;                          // 16 bytes: 4 fp32 or 8 bf16 / fp16
    constexpr int E = U::ELEMS;
    using C = Chunk<U, L::LPN, L::UPL, L::FULLK, false, L::WIDE>;
    using Off_t = typename C::O;
    constexpr int LPN = L::LPN, UPL = L::UPL, G = WAVE / LPN;
    constexpr int NB = C::BIG;                        // steps whose gathers are in flight together
    const int64_t blk = xcd_remap(blockIdx.x, nblocks);
    if (blk < 0) return;
    const int64_t w = blk * waves_in_block() + wave_in_block();
    if (w >= n_items) return;
    const RowItem it = items[w];
    const int row = __builtin_amdgcn_readfirstlane(it.row);
    const int start = __builtin_amdgcn_readfirstlane(it.start);
    const int end = __builtin_amdgcn_readfirstlane(it.end);
    if (start >= end) return;
    const int lane = lane_id();
    const int g = lane / LPN, j = lane & (LPN - 1);
    const Off_t rb = (Off_t)KU * (Off_t)sizeof(T);
    const typename C::Areg a = C::load_a(A, (Off_t)row * rb, j, KU);
    float acc[UPL][E];                                // the lane's units of the output row, fp32
#pragma unroll
    for (int i = 0; i < UPL; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) acc[i][e] = 0.f;
    const int last = end - 1;
    struct Ent { int base, n, c; float s; bool valid; };
    auto entry = [&](int base) {                      // entry base + lane of the item (clamped past its end)
        Ent x;
        x.base = base;
        x.n = base + lane;
        x.valid = x.n < end;
        const int at = x.n < last ? x.n : last;
        x.c = col[at];
        x.s = sval[at];
        return x;
    };
    // steps t0 .. t0+N-1 of a chunk: group g gathers the B rows of entries t*G+g
    auto gather = [&](const Ent &x, int t0, auto &bf) {
        const Off_t boff = (Off_t)x.c * rb;
#pragma unroll
        for (int q = 0; q < (int)(sizeof(bf) / sizeof(bf[0])); ++q) {
            const int src = ((t0 + q) * G + g) & (WAVE - 1);
            const Off_t bo = shfl_off<Off_t>(boff, src);
#pragma unroll
            for (int i = 0; i < UPL; ++i) {
                const int u = C::unit_on(j, i, KU) ? j + i * LPN : 0;
                bf[q][i] = load_at<T, Off_t>(B, bo + (Off_t)(u * (int)sizeof(T)));
            }
        }
    };
    // FULL: all N steps hold entries of the item.  The steps are independent of each other up to the sums into acc: no
    // branch between them, so that their lane exchanges overlap (a branch and a mask per step: graph of 200 000 rows,
    // K = 64 in fp16, 47 us for this kernel, now 37; the whole call 89 -> 83 us; near-dense rows K = 64 46 -> 39 us).
    auto consume = [&](auto full_tag, const Ent &x, int t0, const auto &bf, float &out) {
        constexpr bool FULL = decltype(full_tag)::value;
        constexpr int N = sizeof(bf) / sizeof(bf[0]);
        float p[N];
        bool live[N];
        auto product = [&](int q) {
            const int src = ((t0 + q) * G + g) & (WAVE - 1);
            float d = 0.f;
#pragma unroll
            for (int i = 0; i < UPL; ++i) {
                const float e = U::dot(a.u[i], bf[q][i], d);
                d = C::unit_on(j, i, KU) ? e : d;
            }
            p[q] = group_sum<LPN>(d) * __shfl(x.s, src, WAVE);
            // a step past the end of the row works on a clamped position: it must leave the
            // output row alone whatever that position's B row holds (0 * inf is not 0)
            if constexpr (!FULL) {
                live[q] = x.base + src < end;
                p[q] = live[q] ? p[q] : 0.f;
            }
        };
        auto update = [&](int q) {
#pragma unroll
            for (int i = 0; i < UPL; ++i) {
                float next[E];
#pragma unroll
                for (int e = 0; e < E; ++e) next[e] = acc[i][e];
                U::axpy(p[q], bf[q][i], next);
#pragma unroll
                for (int e = 0; e < E; ++e) acc[i][e] = FULL || live[q] ? next[e] : acc[i][e];
            }
            if (j == t0 + q) out = p[q];
        };
        if constexpr (STEPS) {
            const int steps = (end - x.base + G - 1) / G;
#pragma unroll
            for (int q = 0; q < N; ++q) {
                if (t0 + q >= steps) break;                   // wave-uniform
                product(q);
                update(q);
            }
        } else {
#pragma unroll
            for (int q = 0; q < N; ++q) product(q);
#pragma unroll
            for (int q = 0; q < N; ++q) update(q);
        }
    };
    // entry l = t*G+g was kept by lane g*LPN+t
    auto store_p = [&](const Ent &x, float out) {
        const float res = __shfl(out, (lane % G) * LPN + lane / G, WAVE);
        if (x.valid) P[x.n] = res;
    };
    static_assert(LPN % NB == 0, "whole batches per chunk of 64 entries");
    const std::true_type whole;
    const std::false_type part;
    // the last chunk: whole, half or quarter batches, rounded up
    auto tail = [&](const Ent &x) {
        constexpr int HALF = NB > 1 ? NB / 2 : 1, QUARTER = NB > 3 ? NB / 4 : 1;
        const int steps = (end - x.base + G - 1) / G;
        float out = 0.f;
        for (int t0 = 0; t0 < steps; t0 += NB) {              // wave-uniform
            auto batch = [&](auto n_tag) {
                T bf[decltype(n_tag)::value][UPL];
                gather(x, t0, bf);
                consume(part, x, t0, bf, out);
            };
            const int left = steps - t0;
            if (left > HALF) batch(std::integral_constant<int, NB>{});
            else if (left > QUARTER) batch(std::integral_constant<int, HALF>{});
            else batch(std::integral_constant<int, QUARTER>{});
        }
        store_p(x, out);
    };
    // Whole chunks: the gathers of the next chunk and the indices of the one after it are in flight while a chunk is
    // multiplied, one round trip per chunk.
    // (Rows of more than one unit per lane keep one batch in flight: the second buffer costs them a
    // third of their wavefronts per SIMD, 171 against 153 us on banded rows of 256 bytes.)
    constexpr bool AHEAD = UPL == 1 && NB == LPN;
    Ent cur = entry(start);
    if constexpr (STEPS) {
        Ent nxt = entry(start + WAVE);
        for (int base = start; base < end; base += WAVE) {
            const Ent after = entry(base + 2 * WAVE);
            const int steps = (end - base + G - 1) / G;
            float out = 0.f;
#pragma unroll
            for (int t0 = 0; t0 < LPN; t0 += NB) {
                if (t0 >= steps) break;                       // wave-uniform
                T bf[NB][UPL];
                gather(cur, t0, bf);
                consume(part, cur, t0, bf, out);
            }
            store_p(cur, out);
            cur = nxt;
            nxt = after;
        }
    } else if (end - start >= WAVE) {
        T bcur[NB][UPL];
        if constexpr (AHEAD) gather(cur, 0, bcur);
        Ent nxt = entry(start + WAVE);
        for (int base = start; base + WAVE <= end; base += WAVE) {
            const Ent after = entry(base + 2 * WAVE);
            float out = 0.f;
            if constexpr (AHEAD) {
                T bnxt[NB][UPL];
                if (base + 2 * WAVE <= end) gather(nxt, 0, bnxt);
                consume(whole, cur, 0, bcur, out);
#pragma unroll
                for (int q = 0; q < NB; ++q)
#pragma unroll
                    for (int i = 0; i < UPL; ++i) bcur[q][i] = bnxt[q][i];
            } else {
#pragma unroll 1                                              // (unrolled, the gathers of all batches move to the front)
                for (int t0 = 0; t0 < LPN; t0 += NB) {
                    gather(cur, t0, bcur);
                    consume(whole, cur, t0, bcur, out);
                }
            }
            store_p(cur, out);
            cur = nxt;
            nxt = after;
        }
    }
    if constexpr (!STEPS) {
        if (cur.base < end) tail(cur);
    }
    // add the partial output rows of the G groups: lanes with the same j
#pragma unroll
    for (int off = LPN; off < WAVE; off <<= 1) {
#pragma unroll
        for (int i = 0; i < UPL; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) acc[i][e] += __shfl_xor(acc[i][e], off, WAVE);
    }
    if (g == 0) {
        const int rs = rowptr[row];
        const bool whole_row = start == rs && end == rowptr[row + 1];
        float *orow = (whole_row ? O + (int64_t)row * KU * E : parts + (int64_t)it.extra * KU * E);
        if (!whole_row && start == rs && lane == 0) O[(int64_t)row * KU * E] = __int_as_float(it.extra);
#pragma unroll
        for (int i = 0; i < UPL; ++i) {
            const int u = j + i * LPN;
            if (!C::unit_on(j, i, KU)) continue;
#pragma unroll
            for (int e = 0; e < E; e += 4)
                *reinterpret_cast<float4 *>(orow + E * u + e) =
                    make_float4(acc[i][e], acc[i][e + 1], acc[i][e + 2], acc[i][e + 3]);
        }
    }
}

// Rows of at most max_len entries, one row per lane group: a wavefront takes 64/LPN
// consecutive rows, group g walks row r0+g.  Lane j of a group reads column index and
// S value of entry t0+j, so LPN entries of each row are gathered back to back; the
// P value of entry t0+j ends up in lane j, and the output row needs no reduction
// across groups.  Longer rows are left to k_fusedmm, launched before, and only their pieces
// are added here (rows of more than seg entries).  The rows of 8-row panels (panel_owner[row]
// == 2, when the array is given) are left to the panel kernel: they count as empty and get a
// row of zeros, which that kernel, launched after this one, adds to.  Every row below M has
// its output row written by one or the other, so O needs no clearing before the launches.
template <class L>
__global__ __launch_bounds__(BLOCK) void k_fusedmm_rows(int64_t nblocks, const int32_t *__restrict__ rowptr,
    const unsigned char *__restrict__ panel_owner, const int32_t *__restrict__ col, const float *__restrict__ sval,
    const void *__restrict__ A, const void *__restrict__ B, int KU, float *__restrict__ P, float *__restrict__ O,
    const float *__restrict__ parts, int M, int max_len, int seg) {
    using U = typename L::U;
    using T = typename U::T;
    constexpr int E = U::ELEMS;
    using C = Chunk<U, L::LPN, L::UPL, L::FULLK, false, L::WIDE>;
    using Off_t = typename C::O;
    constexpr int LPN = L::LPN, UPL = L::UPL, G = WAVE / LPN;
    constexpr int NB = C::BIG;
    const int64_t blk = xcd_remap(blockIdx.x, nblocks);
    if (blk < 0) return;
    const int64_t r0 = (blk * waves_in_block() + wave_in_block()) * G;
    if (r0 >= M) return;
    const int lane = lane_id();
    const int g = lane / LPN, j = lane & (LPN - 1);
    const int64_t row = r0 + g;
    int rs = 0, len = 0;
    bool panel = false, is_long = false;              // the panel kernel takes the row, k_fusedmm took it
    if (row < M) {
        rs = rowptr[row];
        len = rowptr[row + 1] - rs;
        panel = panel_owner && panel_owner[row] == 2;
        is_long = len > max_len && !panel;
    }
    add_cut_rows<L>(parts, O, KU, j == 0 && is_long && len > seg, row, len, seg, lane);
    if (panel || is_long) len = 0;
    int longest = len;
    for (int off = LPN; off < WAVE; off <<= 1) {
        const int o = __shfl_xor(longest, off, WAVE);
        longest = o > longest ? o : longest;
    }
    longest = __builtin_amdgcn_readfirstlane(longest);
    const Off_t rb = (Off_t)KU * (Off_t)sizeof(T);
    const typename C::Areg a = C::load_a(A, (Off_t)(row < M ? row : 0) * rb, j, KU);
    float acc[UPL][E];                                // the lane's units of the output row, fp32
#pragma unroll
    for (int i = 0; i < UPL; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) acc[i][e] = 0.f;
    struct Ent { int at, c; float s; bool has; };
    auto entry = [&](int t0) {                        // entry t0 + j of this group's row
        Ent x;
        const int e = t0 + j;
        x.has = e < len;
        x.at = x.has ? rs + e : (len > 0 ? rs + len - 1 : 0);   // a valid position in every lane
        x.c = col[x.at];
        x.s = x.has ? sval[x.at] : 0.f;
        return x;
    };
    auto gather = [&](const Ent &x, int q0, T (&bf)[NB][UPL]) {
        const Off_t boff = (Off_t)x.c * rb;
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const int src = g * LPN + ((q0 + q) & (LPN - 1));
            const Off_t bo = shfl_off<Off_t>(boff, src);
#pragma unroll
            for (int i = 0; i < UPL; ++i) {
                const int u = C::unit_on(j, i, KU) ? j + i * LPN : 0;
                bf[q][i] = load_at<T, Off_t>(B, bo + (Off_t)(u * (int)sizeof(T)));
            }
        }
    };
    auto consume = [&](const Ent &x, int q0, int steps, const T (&bf)[NB][UPL], float &out) {
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            if (q0 + q >= steps) break;               // wave-uniform
            const int src = g * LPN + ((q0 + q) & (LPN - 1));
            float p = 0.f;
#pragma unroll
            for (int i = 0; i < UPL; ++i) {
                const float d = U::dot(a.u[i], bf[q][i], p);
                p = C::unit_on(j, i, KU) ? d : p;
            }
            // a step past the end of the row works on a clamped position: it must leave the
            // output row alone whatever that position's B row holds (0 * inf is not 0)
            const bool live = __shfl((int)x.has, src, WAVE) != 0;
            p = group_sum<LPN>(p) * __shfl(x.s, src, WAVE);   // every lane takes part in the lane exchange
            p = live ? p : 0.f;
#pragma unroll
            for (int i = 0; i < UPL; ++i) {
                float next[E];
#pragma unroll
                for (int e = 0; e < E; ++e) next[e] = acc[i][e];
                U::axpy(p, bf[q][i], next);
#pragma unroll
                for (int e = 0; e < E; ++e) acc[i][e] = live ? next[e] : acc[i][e];
            }
            if (j == q0 + q) out = p;
        }
    };
    // Batches of NB steps, LPN / NB of them per LPN entries of a row: the gathers of the next batch and
    // the indices of the entries after the next LPN are in flight while a batch is multiplied.
    constexpr int BPC = LPN / NB;
    static_assert(LPN % NB == 0, "whole batches per LPN entries");
    constexpr bool AHEAD = UPL <= 2;                 // (rows of more units per lane: measured the same either way)
    Ent cur = entry(0);
    T bcur[NB][UPL];
    if constexpr (AHEAD) {
        if (longest > 0) gather(cur, 0, bcur);                // wave-uniform
    }
    Ent nxt = entry(LPN);
    for (int t0 = 0; t0 < longest; t0 += LPN) {
        const int steps = longest - t0 < LPN ? longest - t0 : LPN;
        const bool more = t0 + LPN < longest;
        const Ent after = entry(t0 + 2 * LPN);
        float out = 0.f;
#pragma unroll
        for (int bq = 0; bq < BPC; ++bq) {
            const int q0 = bq * NB;
            if (q0 >= steps) break;                           // wave-uniform
            if constexpr (AHEAD) {
                T bnxt[NB][UPL];
                if (bq + 1 < BPC && q0 + NB < steps) gather(cur, q0 + NB, bnxt);
                else if (more) gather(nxt, 0, bnxt);
                consume(cur, q0, steps, bcur, out);
#pragma unroll
                for (int q = 0; q < NB; ++q)
#pragma unroll
                    for (int i = 0; i < UPL; ++i) bcur[q][i] = bnxt[q][i];
            } else {
                gather(cur, q0, bcur);
                consume(cur, q0, steps, bcur, out);
            }
        }
        if (cur.has) P[cur.at] = out;
        cur = nxt;
        nxt = after;
    }
    if (row < M && !is_long) {                        // (the accumulators of a panel's row are zero)
        float *orow = O + row * KU * E;
#pragma unroll
        for (int i = 0; i < UPL; ++i) {
            const int u = j + i * LPN;
            if (!C::unit_on(j, i, KU)) continue;
#pragma unroll
            for (int e = 0; e < E; e += 4)
                *reinterpret_cast<float4 *>(orow + E * u + e) =
                    make_float4(acc[i][e], acc[i][e + 1], acc[i][e + 2], acc[i][e + 3]);
        }
    }
}

// The same rows as k_fusedmm_rows when their lengths differ a lot (a power-law graph: most
// rows hold one to three entries, a few dozens): there a lane group that waits for the longest
// of a wavefront's 64/LPN rows idles four steps out of five.  Here a wavefront takes 64
// consecutive rows, numbers their entries across the rows (prefix sum of the lengths, kept in
// LDS with the rows' CSR positions) and deals whole rows out to its lane groups so that every
// group gets about an equal share of the entries.  A group walks its entries LPN at a time: lane
// j finds the row of its entry by bisection over the prefix sums, loads column index and S
// value; step q then takes entry q with all lanes of the group, gathers the entry's A row with
// its B row (the rows change inside a group, as in the flat kernel), and the group's partial
// output row is written whenever the row changes.  Rows without entries of their own (empty,
// left to the panel kernel) get zeros and the pieces of cut rows are added, as in k_fusedmm_rows.
template <class L>
__global__ __launch_bounds__(BLOCK) void k_fusedmm_rows_balanced(int64_t nblocks, const int32_t *__restrict__ rowptr,
    const unsigned char *__restrict__ panel_owner, const int32_t *__restrict__ col, const float *__restrict__ sval,
    const void *__restrict__ A, const void *__restrict__ B, int KU, float *__restrict__ P, float *__restrict__ O,
    const float *__restrict__ parts, int M, int max_len, int seg) {
    using U = typename L::U;
    using T = typename U::T;
    constexpr int E = U::ELEMS;
    using C = Chunk<U, L::LPN, L::UPL, L::FULLK, false, L::WIDE>;
    using Off_t = typename C::O;
    constexpr int LPN = L::LPN, UPL = L::UPL, G = WAVE / LPN;
    constexpr int NB = C::BIG > 4 ? 4 : C::BIG;       // A and B rows of a batch of steps in flight together
    __shared__ int pre_all[WAVES_PER_BLOCK][WAVE], pos_all[WAVES_PER_BLOCK][WAVE];
    const int64_t blk = xcd_remap(blockIdx.x, nblocks);
    if (blk < 0) return;
    const int64_t r0 = (blk * waves_in_block() + wave_in_block()) * WAVE;
    if (r0 >= M) return;
    const int lane = lane_id();
    const int g = lane / LPN, j = lane & (LPN - 1);
    int *pre = pre_all[wave_in_block()], *pos = pos_all[wave_in_block()];
    // lane l: row r0 + l
    const bool inside = r0 + lane < M;
    int rs = 0, len = 0;
    bool panel = false, is_long = false;              // the panel kernel takes the row, k_fusedmm took it
    if (inside) {
        rs = rowptr[r0 + lane];
        len = rowptr[r0 + lane + 1] - rs;
        panel = panel_owner && panel_owner[r0 + lane] == 2;
        is_long = len > max_len && !panel;
    }
    add_cut_rows<L>(parts, O, KU, is_long && len > seg, r0 + lane, len, seg, lane);
    if (panel || is_long) len = 0;
    int incl = len;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const int up = __shfl_up(incl, o, WAVE);
        if (lane >= o) incl += up;
    }
    const int total = __builtin_amdgcn_readlane(incl, WAVE - 1);
    pre[lane] = incl - len;
    pos[lane] = rs;
    wave_lds_order();
    // whole rows per group: group gg starts at the first row whose prefix reaches gg/G of the entries
    int b_lo = 0, b_hi = WAVE;
#pragma unroll
    for (int gg = 1; gg < G; ++gg) {
        const int target = (int)((int64_t)gg * total / G);
        const int first = __popcll(__ballot(incl - len < target));
        if (g == gg) b_lo = first;
        if (g + 1 == gg) b_hi = first;
    }
    const int v_lo = b_lo < WAVE ? pre[b_lo] : total, v_hi = b_hi < WAVE ? pre[b_hi] : total;
    int longest = v_hi - v_lo;
#pragma unroll
    for (int o = LPN; o < WAVE; o <<= 1) {
        const int other = __shfl_xor(longest, o, WAVE);
        longest = other > longest ? other : longest;
    }
    longest = __builtin_amdgcn_readfirstlane(longest);
    const Off_t rb = (Off_t)KU * (Off_t)sizeof(T);
    // rows with nothing of their own: zeros (lane group g takes rows g, g + G, ..)
    {
        const unsigned long long empty = __ballot(inside && len == 0 && !is_long);
#pragma unroll
        for (int k = 0; k < WAVE / G; ++k) {
            const int rr = k * G + g;
            if (!((empty >> rr) & 1ull)) continue;
            float *orow = O + (r0 + rr) * (int64_t)KU * E;
#pragma unroll
            for (int i = 0; i < UPL; ++i) {
                const int u = j + i * LPN;
                if (!C::unit_on(j, i, KU)) continue;
#pragma unroll
                for (int e = 0; e < E; e += 4)
                    *reinterpret_cast<float4 *>(orow + E * u + e) = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    }
    float acc[UPL][E];
#pragma unroll
    for (int i = 0; i < UPL; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) acc[i][e] = 0.f;
    int cur_row = -1;                                 // the row the group's partial sums belong to (the same in its lanes)
    auto flush = [&](bool on) {
        if (!on) return;
        float *orow = O + (r0 + cur_row) * (int64_t)KU * E;
#pragma unroll
        for (int i = 0; i < UPL; ++i) {
            const int u = j + i * LPN;
            if (!C::unit_on(j, i, KU)) continue;
#pragma unroll
            for (int e = 0; e < E; e += 4)
                *reinterpret_cast<float4 *>(orow + E * u + e) =
                    make_float4(acc[i][e], acc[i][e + 1], acc[i][e + 2], acc[i][e + 3]);
        }
    };
    for (int t0 = 0; t0 < longest; t0 += LPN) {
        const int v = v_lo + t0 + j;
        const bool has = v < v_hi;
        // the row of entry v: the last row whose prefix does not exceed v (rows without entries
        // share their prefix with the row after them and are never the last such row)
        const int vv = has ? v : (v_hi > v_lo ? v_hi - 1 : 0);
        int lo = 0, hi = WAVE;
#pragma unroll
        for (int it = 0; it < 6; ++it) {
            const int mid = (lo + hi) >> 1;
            if (pre[mid] <= vv) lo = mid; else hi = mid;
        }
        const int row = v_hi > v_lo ? lo : 0;                            // (a group without entries: row 0, position 0)
        const int at = v_hi > v_lo ? pos[row] + (vv - pre[row]) : 0;      // a valid position in every lane
        const int c = col[at];
        const float s = has ? sval[at] : 0.f;
        const Off_t boff = (Off_t)c * rb, aoff = (Off_t)(r0 + row) * rb;
        const int steps = longest - t0 < LPN ? longest - t0 : LPN;
        float out = 0.f;
        for (int q0 = 0; q0 < steps; q0 += NB) {
            T bf[NB][UPL], af[NB][UPL];
#pragma unroll
            for (int q = 0; q < NB; ++q) {
                const int src = g * LPN + ((q0 + q) & (LPN - 1));
                const Off_t bo = shfl_off<Off_t>(boff, src), ao = shfl_off<Off_t>(aoff, src);
#pragma unroll
                for (int i = 0; i < UPL; ++i) {
                    const int u = C::unit_on(j, i, KU) ? j + i * LPN : 0;
                    bf[q][i] = load_at<T, Off_t>(B, bo + (Off_t)(u * (int)sizeof(T)));
                    af[q][i] = load_at<T, Off_t>(A, ao + (Off_t)(u * (int)sizeof(T)));
                }
            }
#pragma unroll
            for (int q = 0; q < NB; ++q) {
                if (q0 + q >= steps) break;               // wave-uniform
                const int src = g * LPN + ((q0 + q) & (LPN - 1));
                const bool live = __shfl((int)has, src, WAVE) != 0;
                const int row_q = __shfl(row, src, WAVE);
                const bool change = live && row_q != cur_row;
                flush(change && cur_row >= 0);
                cur_row = change ? row_q : cur_row;
                float p = 0.f;
#pragma unroll
                for (int i = 0; i < UPL; ++i) {
                    const float d = U::dot(af[q][i], bf[q][i], p);
                    p = C::unit_on(j, i, KU) ? d : p;
                }
                // a step past the end of the group's entries works on a clamped position: it must leave
                // the output row alone whatever that position's B row holds (0 * inf is not 0)
                p = group_sum<LPN>(p) * __shfl(s, src, WAVE);     // every lane takes part in the lane exchange
                p = live ? p : 0.f;
#pragma unroll
                for (int i = 0; i < UPL; ++i) {
                    float next[E];
#pragma unroll
                    for (int e = 0; e < E; ++e) next[e] = change ? 0.f : acc[i][e];
                    U::axpy(p, bf[q][i], next);
#pragma unroll
                    for (int e = 0; e < E; ++e) acc[i][e] = live ? next[e] : acc[i][e];
                }
                if (j == q0 + q) out = p;
            }
        }
        if (has) P[at] = out;
    }
    flush(cur_row >= 0);
}

}  // namespace sddmm
