// Operands staged through registers: the kernels whose operands the LDS DMA
// cannot take (suffix _u: rows that are not 16-byte aligned).
//
// Included by gemm_gfx950.hip after its DMA operands, whose LDS layouts, swizzles
// and fragment reads are used unchanged: a stage holds 64 K values of both
// tiles, and a thread's piece is one 16-byte slot of it (8 bf16 along the
// operand's contiguous dimension).  Here the piece comes through VGPRs: a
// 16-byte global load at any 2-byte address (gfx950 runs in unaligned access
// mode), kept in flight for D stages, then one ds_write_b128.
//
// What bounds it: the step's chain of LDS reads, LDS writes and a barrier with one
// or two workgroups per CU; the D stages in flight (4 for 64x64, 2 for 128x128,
// whose registers allow no more with two workgroups per CU) cover the memory
// latency.  1001 x 1003 x 999: NT 36.3 -> 10.3 us, TN 172.6 -> 10.5 us against
// element-wise loads, eight per piece, with one stage in flight; 4097^3 NT
// 1853 -> 272 us.
#ifndef T0G_GEMM_STAGED_H
#define T0G_GEMM_STAGED_H

namespace t0g {

typedef const __attribute__((address_space(1))) char gbytes_t;
// 16 bytes at any element address
typedef u32x4_t __attribute__((aligned(2))) u32x4_u_t;

__device__ __forceinline__ u32x4_t load16_u(gbytes_t* p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) u32x4_u_t*>(p);
}

// 8 bf16 moved down by `s` elements (0 .. 8), zeros filling the top.
__device__ __forceinline__ u32x4_t shift_down8(u32x4_t v, uint32_t s) {
    uint64_t lo = (uint64_t)v[0] | ((uint64_t)v[1] << 32), hi = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
    if (s >= 4) {
        lo = hi;
        hi = 0;
        s -= 4;
    }
    if (s >= 4) {
        lo = 0;
        s = 0;
    }
    const uint32_t b = s * 16;
    lo = (lo >> b) | ((hi << 1) << (63 - b));
    hi >>= b;
    return u32x4_t{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// The pieces of one operand.  Rows (K-contiguous) or columns (M/N-contiguous)
// past the operand read some element inside it: their products are never
// stored.  K values at or past kend read as zero.
//
// A stage is whole or an edge stage (uniform, the same for both operands):
//   whole: every piece is 8 values of the operand's memory.  For an
//     M/N-contiguous operand a piece at the ragged edge runs into the next k
//     row, which is memory of the operand as long as one follows (whole());
//   edge (the last stage, as a rule): pieces start no later than 8 values before
//     the end of their row (K range or columns) and are shifted into place, so
//     nothing past the row is read; rows of fewer than 8 values are read element
//     by element.
template <bool K_MAJOR, int ROWS, int NT, int SUBS>
struct StagedOperand : DmaOperand<K_MAJOR, ROWS, NT, SUBS, 64> {
    typedef DmaOperand<K_MAJOR, ROWS, NT, SUBS, 64> Dma;
    static constexpr int kInstr = Dma::kInstr;
    uint32_t rowb[kInstr];   // byte offset of the piece's row (K-contiguous) or of its k row at k0 = 0
    uint32_t pos[kInstr];    // K-contiguous: K column within the stage; M/N-contiguous: column of the operand
    uint32_t rows;           // M/N rows of the operand
    uint32_t last_col;       // M/N-contiguous: the tile's last piece's column

    __device__ __forceinline__ void init(uint32_t tid, uint32_t row0, uint32_t R, uint32_t ld, uint32_t wrow, uint32_t l32,
                                         uint32_t g) {
        Dma::init(tid, row0, ld, wrow, l32, g);
        rows = R;
        last_col = row0 + ROWS - 8;
        const uint32_t lane = tid & 63u;
#pragma unroll
        for (int i = 0; i < kInstr; ++i) {
            if constexpr (K_MAJOR) {
                const uint32_t r = row0 + Dma::kRowsPerInstr * (i * Dma::kWaves + this->wave) + lane / Dma::kChunks;
                rowb[i] = (r < R ? r : R - 1) * ld * 2;
                pos[i] = this->kcol[i];
            } else {
                const uint32_t slot = ((i * Dma::kWaves + this->wave) * 1024 + lane * 16) % Dma::kRowB / 16;
                const uint32_t lg = (slot >> 1) ^ fm(this->krow[i], Dma::kGranules);
                rowb[i] = this->krow[i] * ld * 2;
                pos[i] = row0 + lg * 16 + (slot & 1) * 8;
            }
        }
    }
    __device__ __forceinline__ uint32_t k_row(int i) const {
        if constexpr (K_MAJOR) return 0u;
        else return this->krow[i];
    }
    // Whether the stage at k0 (64 K values inside the K range) is whole.
    __device__ __forceinline__ bool whole(uint32_t k0, uint32_t ld, uint32_t k) const {
        if constexpr (K_MAJOR) return true;
        // the last piece of k row k0 + 63 ends inside the operand
        const uint32_t c = last_col < rows - 1 ? last_col : rows - 1;
        return (k - 64 - k0) * ld + rows >= c + 8;
    }
    __device__ __forceinline__ void load_whole(u32x4_t (&v)[kInstr], uint64_t base, uint32_t ld, uint32_t k0) const {
        // kept scalar: the loads add their 32-bit offsets to it
        const uint64_t b = base + (K_MAJOR ? (uint64_t)k0 * 2 : (uint64_t)k0 * ld * 2);
        gbytes_t* p = reinterpret_cast<gbytes_t*>(((uint64_t)uniform_u32((uint32_t)(b >> 32)) << 32) | uniform_u32((uint32_t)b));
#pragma unroll
        for (int i = 0; i < kInstr; ++i) {
            uint32_t o = rowb[i] + (K_MAJOR || pos[i] < rows ? pos[i] : rows - 1) * 2;
            asm("" : "+v"(o));   // a 32-bit offset again in every step, not a 64-bit address
            v[i] = load16_u(p + o);
        }
    }
    // Edge stage: fetch sends the loads, finish puts the values in place.
    __device__ __forceinline__ uint32_t row_end(uint32_t kend) const { return K_MAJOR ? kend : rows; }
    __device__ __forceinline__ void fetch_edge(u32x4_t (&v)[kInstr], uint64_t base, uint32_t ld, uint32_t k0,
                                               uint32_t kend) const {
        gbytes_t* p = reinterpret_cast<gbytes_t*>(base);
        const uint32_t end = row_end(kend);
#pragma unroll
        for (int i = 0; i < kInstr; ++i) {
            const uint32_t k = K_MAJOR ? 0u : k0 + k_row(i);
            const uint32_t rb = K_MAJOR ? rowb[i] : (k < kend ? k : kend - 1) * ld * 2;
            const uint32_t at = K_MAJOR ? k0 + pos[i] : pos[i];
            if (end >= 8) {
                v[i] = load16_u(p + (rb + (at < end - 8 ? at : end - 8) * 2));
            } else {
                uint16_t e[8];
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j) {
                    const uint32_t x = at + j < end ? at + j : end - 1;
                    const uint16_t t = *reinterpret_cast<gu16_t*>(p + (rb + x * 2));
                    e[j] = at + j < end ? t : (uint16_t)0;
                }
                v[i] = pack8(e);
            }
        }
    }
    __device__ __forceinline__ void finish_edge(u32x4_t (&v)[kInstr], uint32_t k0, uint32_t kend) const {
        const uint32_t end = row_end(kend);
#pragma unroll
        for (int i = 0; i < kInstr; ++i) {
            if (end >= 8) {
                const uint32_t at = K_MAJOR ? k0 + pos[i] : pos[i];
                const uint32_t s = at < end - 8 ? 0u : at - (end - 8);
                v[i] = shift_down8(v[i], s < 8 ? s : 8);
            }
            if (!K_MAJOR && k0 + k_row(i) >= kend) v[i] = zero4();
        }
    }
    __device__ __forceinline__ void commit(const u32x4_t (&v)[kInstr], uint32_t lds) const {
        typedef __attribute__((address_space(3))) u32x4_t lds_u32x4;
        const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
        for (int i = 0; i < kInstr; ++i)
            *reinterpret_cast<lds_u32x4*>((uintptr_t)(lds + (i * Dma::kWaves + this->wave) * 1024 + lane * 16)) = v[i];
    }
};

// K loop: two LDS stages of 64 K values, D stages of pieces in VGPRs.  Step s
// writes stage s + 1 (loaded D steps ago) to the buffer stage s - 1 freed at
// the last barrier, sends the loads of stage s + 1 + D, and multiplies stage s.
// The loop takes the whole stages only and always sends its loads (past the
// end: stage 0's again, which is in the caches): with a choice of load paths
// inside, the compiler waits for more than the stage it needs.  The edge
// stage's loads go out first and are put in place after the loop.
template <int D, uint32_t A_BYTES, uint32_t STAGE, int SM, int SN, class OpA, class OpB>
__device__ __forceinline__ void k_pipeline_staged(f32x16_t (&acc)[SM][SN], const OpA& la, const OpB& lb,
                                                  const T0gGemmArgs& p, uint32_t kbeg, uint32_t kend, int nst,
                                                  uint32_t lds0) {
    static_assert(D % 2 == 0, "the LDS buffer of a step is its parity");
    int nw = (int)((kend - kbeg) / 64);   // leading whole stages
    while (nw > 0 && !(la.whole(kbeg + (uint32_t)(nw - 1) * 64, p.lda, p.k) &&
                       lb.whole(kbeg + (uint32_t)(nw - 1) * 64, p.ldb, p.k)))
        --nw;
    auto barrier = [&] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        barrier_no_fence();
    };
    u32x4_t ea[OpA::kInstr], eb[OpB::kInstr];
    if (nw < nst) {
        la.fetch_edge(ea, p.a, p.lda, kbeg + (uint32_t)nw * 64, kend);
        lb.fetch_edge(eb, p.b, p.ldb, kbeg + (uint32_t)nw * 64, kend);
    }
    uint32_t cur = lds0;
    if (nw > 0) {
        u32x4_t va[D][OpA::kInstr], vb[D][OpB::kInstr];
        auto load = [&](int t, u32x4_t (&a)[OpA::kInstr], u32x4_t (&b)[OpB::kInstr]) {
            const uint32_t k0 = kbeg + (uint32_t)(t < nw ? t : 0) * 64;
            la.load_whole(a, p.a, p.lda, k0);
            lb.load_whole(b, p.b, p.ldb, k0);
        };
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load(d, va[d], vb[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
        la.commit(va[0], lds0);
        lb.commit(vb[0], lds0 + A_BYTES);
        load(D, va[0], vb[0]);
        barrier();
        // step u (mod D): stage s + u from its buffer; the next stage's pieces to the other
        auto step = [&](int u, int t_load, bool send) {
            const uint32_t st = lds0 + (u & 1) * STAGE, nxt = lds0 + ((u + 1) & 1) * STAGE;
            bf16x8_t fa[2][SM], fb[2][SN];
            la.template read<0>(st, fa[0]);
            lb.template read<0>(st + A_BYTES, fb[0]);
            la.template read<1>(st, fa[1]);
            lb.template read<1>(st + A_BYTES, fb[1]);
            la.commit(va[(u + 1) % D], nxt);
            lb.commit(vb[(u + 1) % D], nxt + A_BYTES);
            if (send) load(t_load, va[(u + 1) % D], vb[(u + 1) % D]);
            mfma_step(acc, fa[0], fb[0]);
            la.template read<2>(st, fa[0]);
            lb.template read<2>(st + A_BYTES, fb[0]);
            mfma_step(acc, fa[1], fb[1]);
            la.template read<3>(st, fa[1]);
            lb.template read<3>(st + A_BYTES, fb[1]);
            mfma_step(acc, fa[0], fb[0]);
            mfma_step(acc, fa[1], fb[1]);
            barrier();
        };
        // whole rounds of D steps with one exit (the compiler joins several exits of a
        // loop into its latch, and the wait counts at its top must hold for all of
        // them), then the rest, whose stages are all in flight already
        const int rounds = nw / D, rest = nw % D;
        for (int r = 0; r < rounds; ++r)
#pragma unroll
            for (int u = 0; u < D; ++u) step(u, r * D + u + 1 + D, true);
#pragma unroll
        for (int u = 0; u < D - 1; ++u)
            if (u < rest) step(u, 0, false);
        // the last step wrote a stage past the end to the next buffer, which nobody reads
        cur = lds0 + ((uint32_t)nw & 1u) * STAGE;
    }
    for (int s = nw; s < nst; ++s) {
        const uint32_t k0 = kbeg + (uint32_t)s * 64;
        if (s > nw) {
            la.fetch_edge(ea, p.a, p.lda, k0, kend);
            lb.fetch_edge(eb, p.b, p.ldb, k0, kend);
        }
        la.finish_edge(ea, k0, kend);
        lb.finish_edge(eb, k0, kend);
        la.commit(ea, cur);
        lb.commit(eb, cur + A_BYTES);
        barrier();
        bf16x8_t fa[SM], fb[SN];
        la.template read<0>(cur, fa);
        lb.template read<0>(cur + A_BYTES, fb);
        mfma_step(acc, fa, fb);
        la.template read<1>(cur, fa);
        lb.template read<1>(cur + A_BYTES, fb);
        mfma_step(acc, fa, fb);
        la.template read<2>(cur, fa);
        lb.template read<2>(cur + A_BYTES, fb);
        mfma_step(acc, fa, fb);
        la.template read<3>(cur, fa);
        lb.template read<3>(cur + A_BYTES, fb);
        mfma_step(acc, fa, fb);
        cur = cur == lds0 ? lds0 + STAGE : lds0;   // the other buffer's readers passed this step's barrier
    }
}

template <int BM, int BN, int WAVES_M, int WAVES_N, bool A_K, bool B_K, bool OUT_BF16, int D>
__device__ __forceinline__ void gemm_tile_staged(const T0gGemmArgs& p) {
    constexpr int NT = 64 * WAVES_M * WAVES_N;
    constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
    constexpr int SM = WTM / 32, SN = WTN / 32;
    using OpA = StagedOperand<A_K, BM, NT, SM>;
    using OpB = StagedOperand<B_K, BN, NT, SN>;
    constexpr uint32_t A_BYTES = OpA::kStageBytes, STAGE = OpA::kStageBytes + OpB::kStageBytes;
    __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];

    const uint32_t tid = threadIdx.x;
    const GridPos gp = grid_pos(p);
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
    const uint32_t wm = wave / WAVES_N, wn = wave % WAVES_N;
    const uint32_t l32 = lane & 31u, g = lane >> 5;
    f32x16_t acc[SM][SN];
#pragma unroll
    for (int i = 0; i < SM; ++i)
#pragma unroll
        for (int j = 0; j < SN; ++j) acc[i][j] = f32x16_t{};
    if (nst > 0) {
        OpA la;
        OpB lb;
        la.init(tid, m0, p.m, p.lda, wm * WTM, l32, g);
        lb.init(tid, n0, p.n, p.ldb, wn * WTN, l32, g);
        k_pipeline_staged<D, A_BYTES, STAGE>(acc, la, lb, p, kbeg, kend, nst,
                                             __builtin_amdgcn_readfirstlane(lds_addr(smem)));
    }
    store_tile<SM, SN, OUT_BF16>(p, acc, m0 + wm * WTM, n0 + wn * WTN, l32, g, gp.split);
}

}  // namespace t0g

#endif
