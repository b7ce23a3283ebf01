// Operands staged through registers: the kernels whose operands the LDS DMA
// cannot take -- bf16 rows that are not 16-byte aligned (suffix _u), f32 operands
// that are rounded to bf16 on the way (_ff, _fb).
//
// Included by gemm_gfx950.hip after its DMA operands, whose LDS layouts, swizzles,
// fragment reads and K loops are used unchanged: a stage holds 64 K values of both
// tiles.  Here its pieces come through VGPRs: a 16-byte global load at any element
// address (gfx950 runs in unaligned access mode), kept in flight for D stages, then
// an LDS write.  Four waves stage, four multiply, one of each per SIMD, so a piece's
// rounding and address arithmetic run beside the MFMAs.
//
// What bounds it: the loads into one CU (a 64x64 step takes 0.33 us with 16 KB of
// bf16 or one f32 operand, 0.5 us with two: 32 KB); the element-wise loads before
// were bound by their count, eight 2-byte loads per piece with one stage in flight.
// 1001 x 1003 x 999: NT 36.3 -> 10.0 us, TN 172.6 -> 10.3 us; 4097^3 NT 1853 -> 250 us.
// f32 1024^3 forward 15.9 -> 12.1 us, 32 x 128 x 128 10.0 -> 4.5 us against two
// conversion launches and the bf16 GEMM.
#ifndef T0G_GEMM_STAGED_H
#define T0G_GEMM_STAGED_H

namespace t0g {

typedef const __attribute__((address_space(1))) char gbytes_t;
// 16 bytes at any element address
__device__ __forceinline__ u32x4_t load16_any(gbytes_t* p) {
    typedef u32x4_t __attribute__((aligned(2))) u32x4_any_t;
    return *reinterpret_cast<const __attribute__((address_space(1))) u32x4_any_t*>(p);
}

// 16 bytes moved down by `s` bytes (even, 0 .. 16), zeros filling the top.
__device__ __forceinline__ u32x4_t shift_down16(u32x4_t v, uint32_t s) {
    uint64_t lo = (uint64_t)v[0] | ((uint64_t)v[1] << 32), hi = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
    if (s >= 8) {
        lo = hi;
        hi = 0;
        s -= 8;
    }
    if (s >= 8) {
        lo = 0;
        s = 0;
    }
    const uint32_t b = s * 8;
    lo = (lo >> b) | ((hi << 1) << (63 - b));
    hi >>= b;
    return u32x4_t{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// The pieces of one operand: 16 bytes of memory each, 8 bf16 or (F32) 4 f32,
// which commit() rounds to bf16 with the operand conversion's rounding
// (t0g_f32_to_bf16_rne).  A wave's pieces fill consecutive LDS slots, so its lanes
// read whole consecutive cache lines.  Rows (K-contiguous) or columns
// (M/N-contiguous) past the operand read some element inside it: their products
// are never stored.  K values at or past kend read as zero.
//
// A stage is whole or an edge stage (uniform, the same for both operands):
//   whole: every piece is 16 bytes of the operand's memory.  For an
//     M/N-contiguous operand a piece across the ragged edge runs into the next k
//     row, which is memory of the operand as long as one follows (whole());
//   edge (the last stage, as a rule): pieces start no later than one piece before
//     the end of their row (K range or columns) and are shifted into place, so
//     nothing past the row is read; rows shorter than a piece are read element by
//     element.
template <bool K_MAJOR, int ROWS, int NT, int SUBS, bool F32 = false>
struct StagedOperand {
    typedef DmaOperand<K_MAJOR, ROWS, NT, SUBS, 64> Dma;
    static constexpr uint32_t kSize = F32 ? 4 : 2;         // bytes of an element
    static constexpr uint32_t kVals = 16 / kSize;          // elements of a piece
    static constexpr uint32_t kSlot = 2 * kVals;           // its bytes in LDS
    static constexpr int kPieces = ROWS * 64 / (int)kVals / NT;
    typedef u32x4_t pieces_t[kPieces];
    uint32_t off[kPieces];    // byte offset of the piece at k0 = 0 (pieces past the operand moved inside)
    uint32_t row0, rows;      // the tile's first M/N row, the operand's M/N rows
    uint32_t last_col;        // M/N-contiguous: the furthest column a piece of the tile starts at
    uint32_t slot;            // LDS offset of the lane's piece 0 in a stage

    // Piece i of thread tid: its M/N row (K-contiguous) or k row within the stage, and
    // its K column within the stage or its column of the operand.
    struct Where {
        uint32_t row, col;
    };
    __device__ __forceinline__ Where where(uint32_t tid, int i) const {
        const uint32_t at = (tid + i * NT) * kSlot;   // byte in the stage
        const uint32_t in16 = at % 16 / 2;            // element within a 16-byte chunk
        if constexpr (K_MAJOR) {
            const uint32_t r = at / Dma::kKRow, c = (at % Dma::kKRow / 16) ^ fk<64>(r);
            return Where{row0 + r < rows ? row0 + r : rows - 1, c * 8 + in16};
        } else {
            const uint32_t k = at / Dma::kRowB, s = at % Dma::kRowB / 16;
            const uint32_t lg = (s >> 1) ^ fm(k, Dma::kGranules);
            return Where{k, row0 + lg * 16 + (s & 1) * 8 + in16};
        }
    }
    __device__ __forceinline__ void init(uint32_t tid, uint32_t first, uint32_t R, uint32_t ld) {
        row0 = first;
        rows = R;
        const uint32_t outside = R >= kVals ? R - kVals : 0;   // columns read by pieces wholly past the operand
        last_col = min(row0 + ROWS - kVals, (R - 1) & ~(kVals - 1));   // not below `outside` where that is read
        slot = tid * kSlot;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const Where w = where(tid, i);
            off[i] = (w.row * ld + (K_MAJOR || w.col < rows ? w.col : outside)) * kSize;
        }
    }
    // Whether the stage at k0 (64 K values inside the K range) is whole.
    __device__ __forceinline__ bool whole(uint32_t k0, uint32_t ld, uint32_t k) const {
        if constexpr (K_MAJOR) return true;
        // the furthest piece of k row k0 + 63 ends inside the operand
        return (k - 64 - k0) * ld + rows >= last_col + kVals;
    }
    __device__ __forceinline__ void load_whole(pieces_t& v, uint64_t base, uint32_t ld, uint32_t k0) const {
        // kept scalar: the loads add their 32-bit offsets to it
        const uint64_t b = base + (K_MAJOR ? (uint64_t)k0 * kSize : (uint64_t)k0 * ld * kSize);
        gbytes_t* p = reinterpret_cast<gbytes_t*>(((uint64_t)uniform_u32((uint32_t)(b >> 32)) << 32) | uniform_u32((uint32_t)b));
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            uint32_t o = off[i];
            asm("" : "+v"(o));   // a 32-bit offset again in every step, not a 64-bit address
            v[i] = load16_any(p + o);
        }
    }
    // Edge stage: fetch sends the loads, finish puts the values in place.  Both work
    // the pieces' places out again from an opaque thread id, so that nothing of them
    // is held in registers across the loop.
    __device__ __forceinline__ void fetch_edge(pieces_t& v, uint64_t base, uint32_t ld, uint32_t k0, uint32_t kend) const {
        gbytes_t* p = reinterpret_cast<gbytes_t*>(base);
        const uint32_t end = K_MAJOR ? kend : rows;   // one past the row's last value
        const uint32_t tid = opaque_tid() % NT;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const Where w = where(tid, i);
            const uint32_t k = k0 + w.row;
            gbytes_t* row = p + (K_MAJOR ? w.row : (k < kend ? k : kend - 1)) * ld * kSize;
            const uint32_t at = K_MAJOR ? k0 + w.col : w.col;
            if (end >= kVals) {
                v[i] = load16_any(row + (at < end - kVals ? at : end - kVals) * kSize);
            } else {
#pragma unroll
                for (uint32_t j = 0; j < kVals; ++j) {
                    gbytes_t* e = row + (at + j < end ? at + j : end - 1) * kSize;
                    if constexpr (F32)
                        v[i][j] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t*>(e);
                    else if (j % 2 == 0)
                        v[i][j / 2] = *reinterpret_cast<gu16_t*>(e);
                    else
                        v[i][j / 2] |= (uint32_t)*reinterpret_cast<gu16_t*>(e) << 16;
                }
            }
        }
    }
    __device__ __forceinline__ void finish_edge(pieces_t& v, uint32_t k0, uint32_t kend) const {
        const uint32_t end = K_MAJOR ? kend : rows;
        const uint32_t tid = opaque_tid() % NT;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const Where w = where(tid, i);
            const uint32_t at = K_MAJOR ? k0 + w.col : w.col;
            if (end >= kVals) {
                const uint32_t s = at < end - kVals ? 0u : at - (end - kVals);
                v[i] = shift_down16(v[i], (s < kVals ? s : kVals) * kSize);
            } else {
                // a K row's tail becomes zero; past a column edge the value does not matter
                const uint32_t n = (at < end ? end - at : 0u) * kSize;   // bytes kept
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    v[i][j] = 4 * j + 4 <= n ? v[i][j] : 4 * j < n ? v[i][j] & 0xFFFFu : 0u;
            }
            if (!K_MAJOR && k0 + w.row >= kend) v[i] = zero4();
        }
    }
    __device__ __forceinline__ void commit(const pieces_t& v, uint32_t lds) const {
        typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(3))) u32x2_t lds_u32x2;
        typedef __attribute__((address_space(3))) u32x4_t lds_u32x4;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const uintptr_t at = lds + slot + (uint32_t)i * NT * kSlot;
            if constexpr (F32) {
                u32x2_t w;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint32_t lo = v[i][2 * j], hi = v[i][2 * j + 1];
                    const uint32_t rl = lo + 0x7FFFu + ((lo >> 16) & 1u), rh = hi + 0x7FFFu + ((hi >> 16) & 1u);
                    w[j] = __builtin_amdgcn_perm(rh, rl, 0x07060302u);   // the upper halves
                }
                *reinterpret_cast<lds_u32x2*>(at) = w;
            } else {
                *reinterpret_cast<lds_u32x4*>(at) = v[i];
            }
        }
    }
};

// The staging half of a kernel, run by four waves of their own next to the four
// MFMA waves (one of each per SIMD): a ring of three LDS stages of 64 K values
// and D stages of pieces in VGPRs.  While the MFMA waves multiply stage s and read
// the fragments of stage s + 1, step s writes stage s + 2 (loaded D steps ago),
// sends the loads of stage s + 2 + D and meets them at the step's barrier: nst
// barriers after the one that makes stages 0 and 1 visible.
// The loop takes whole stages only, with one exit, and always sends its loads
// (past the end: stage 0's again, which is in the caches): with a choice of load
// paths inside, or several exits, which the compiler joins into the latch, the
// wait counts at its top have to hold for every joined path and wait for more
// than the stage needed.  The edge stage's loads go out first.
template <int D, uint32_t A_BYTES, uint32_t STAGE, class OpA, class OpB>
__device__ __forceinline__ void staged_feed(const OpA& la, const OpB& lb, const T0gGemmArgs& p, uint32_t kbeg,
                                            uint32_t kend, int nst, uint32_t lds0) {
    static_assert(D >= 2, "stages 0 and 1 are written before the loop");
    int nw = (int)((kend - kbeg) / 64);   // leading whole stages
    while (nw > 0 && !(la.whole(kbeg + (uint32_t)(nw - 1) * 64, p.lda, p.k) &&
                       lb.whole(kbeg + (uint32_t)(nw - 1) * 64, p.ldb, p.k)))
        --nw;
    auto barrier = [&] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        barrier_no_fence();
    };
    typename OpA::pieces_t ea, va[D];
    typename OpB::pieces_t eb, vb[D];
    auto fetch = [&](int t) {
        la.fetch_edge(ea, p.a, p.lda, kbeg + (uint32_t)t * 64, kend);
        lb.fetch_edge(eb, p.b, p.ldb, kbeg + (uint32_t)t * 64, kend);
    };
    auto load = [&](int t, typename OpA::pieces_t& a, typename OpB::pieces_t& b) {
        const uint32_t k0 = kbeg + (uint32_t)(t < nw ? t : 0) * 64;
        la.load_whole(a, p.a, p.lda, k0);
        lb.load_whole(b, p.b, p.ldb, k0);
    };
    uint32_t fill = lds0;   // buffer of the next stage to write
    auto commit = [&](const typename OpA::pieces_t& a, const typename OpB::pieces_t& b) {
        la.commit(a, fill);
        lb.commit(b, fill + A_BYTES);
        fill = fill + STAGE == lds0 + 3 * STAGE ? lds0 : fill + STAGE;
    };
    auto edge = [&](int t) {
        if (t > nw) fetch(t);   // only M/N-contiguous rows of fewer than 8 values have a second one
        la.finish_edge(ea, kbeg + (uint32_t)t * 64, kend);
        lb.finish_edge(eb, kbeg + (uint32_t)t * 64, kend);
        commit(ea, eb);
    };
    if (nw < nst) fetch(nw);
    if (nw >= 2) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load(d, va[d], vb[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
        commit(va[0], vb[0]);
        load(D, va[0], vb[0]);
        commit(va[1], vb[1]);
        load(D + 1, va[1], vb[1]);
        barrier();
        const int rounds = (nw - 2) / D, rest = (nw - 2) % D;
        for (int r = 0; r < rounds; ++r)
#pragma unroll
            for (int u = 0; u < D; ++u) {
                commit(va[(2 + u) % D], vb[(2 + u) % D]);
                load(2 + r * D + u + D, va[(2 + u) % D], vb[(2 + u) % D]);
                barrier();
            }
#pragma unroll
        for (int u = 0; u < D - 1; ++u)
            if (u < rest) {
                commit(va[(2 + u) % D], vb[(2 + u) % D]);
                barrier();
            }
        for (int t = nw; t < nst; ++t) {
            edge(t);
            barrier();
        }
    } else {
        // at most one whole stage
        for (int t = 0; t < nst; ++t) {
            if (t < nw) {
                load(t, va[0], vb[0]);
                commit(va[0], vb[0]);
            } else {
                edge(t);
            }
            if (t >= 1 || nst == 1) barrier();   // stages 0 and 1 share the first barrier
        }
    }
    // the last two steps have nothing left to write
    barrier();
    if (nst >= 2) barrier();
}

template <int BM, int BN, bool A_K, bool B_K, bool OUT_BF16, int D, bool A_F32 = false, bool B_F32 = false>
__device__ __forceinline__ void gemm_tile_staged(const T0gGemmArgs& p) {
    constexpr int NT = 256;   // MFMA threads, and as many staging threads
    constexpr int WTM = BM / 2, WTN = BN / 2;
    constexpr int SM = WTM / 32, SN = WTN / 32;
    using OpA = StagedOperand<A_K, BM, NT, SM, A_F32>;
    using OpB = StagedOperand<B_K, BN, NT, SN, B_F32>;
    constexpr uint32_t A_BYTES = OpA::Dma::kStageBytes, STAGE = A_BYTES + OpB::Dma::kStageBytes;
    __shared__ __attribute__((aligned(1024))) char smem[3 * STAGE];

    const uint32_t tid = threadIdx.x % NT;
    const GridPos gp = grid_pos<true>(p);
    const uint32_t gm = p.group_m;
    const uint32_t per_group = gm * p.tiles_n;
    const uint32_t group = gp.tile / per_group;
    const uint32_t first_m = group * gm;
    const uint32_t gsz = min(p.tiles_m - first_m, gm);
    const uint32_t in_group = gp.tile - group * per_group;
    const uint32_t m0 = (first_m + in_group % gsz) * BM;
    const uint32_t n0 = (in_group / gsz) * BN;

    const uint32_t kbeg = gp.split * p.k_per_split;
    const uint32_t kend = min(p.k, kbeg + p.k_per_split);
    const int nst = kend > kbeg ? (int)((kend - kbeg + 63) / 64) : 0;

    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t wm = wave / 2, wn = wave % 2;
    const uint32_t l32 = lane & 31u, g = lane >> 5;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem));
    const bool stager = __builtin_amdgcn_readfirstlane(threadIdx.x) >= NT;
    if (stager) {
        if (nst > 0) {
            OpA la;
            OpB lb;
            la.init(tid, m0, p.m, p.lda);
            lb.init(tid, n0, p.n, p.ldb);
            staged_feed<D, A_BYTES, STAGE>(la, lb, p, kbeg, kend, nst, lds0);
        }
        return;
    }
    // 64x64: even and odd K steps are summed apart and added at the end.  It costs 16
    // registers and no time, and a K range that the fast path would cut over its waves
    // keeps that path's error (512 x 768 x 3072: 1.3e-7 of the result).
    constexpr int NACC = SM * SN == 1 ? 2 : 1;
    f32x16_t acc[NACC][SM][SN];
#pragma unroll
    for (int a = 0; a < NACC; ++a)
#pragma unroll
        for (int i = 0; i < SM; ++i)
#pragma unroll
            for (int j = 0; j < SN; ++j) acc[a][i][j] = f32x16_t{};
    if (nst > 0) {
        typename OpA::Dma la;
        typename OpB::Dma lb;
        la.init(tid, m0, p.lda, wm * WTM, l32, g);
        lb.init(tid, n0, p.ldb, wn * WTN, l32, g);
        if constexpr (NACC == 2) {
            k_pipeline_deep<false, false, 3, A_BYTES, STAGE, 0>(acc, la, lb, p, 0u, 0u, kbeg, kend, nst, lds0);
            acc[0][0][0] += acc[1][0][0];
        } else {
            k_pipeline<false, false, 64, 3, A_BYTES, STAGE, 0>(acc[0], la, lb, p, 0u, 0u, kbeg, kend, nst, lds0);
        }
    }
    store_tile<SM, SN, OUT_BF16>(p, acc[0], m0 + wm * WTM, n0 + wn * WTN, l32, g, gp.split);
}

}  // namespace t0g

#endif
