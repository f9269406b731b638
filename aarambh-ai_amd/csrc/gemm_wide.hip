// Quantised GEMM with wide wave tiles on gfx950: INT4 projections and the BF16 LM head where
// the row and column blocks fill the part without k-splits (gemm_wide_wins).  Same operands,
// products and epilogues as gemm.hip (QatLinear::forward, quant/src/qat.rs:315-348).
//
// What bounds gemm.hip's loop is a wave tile of 32 rows: each dequantised INT4 word (9 VALU
// operations) feeds four MFMAs, while a SIMD that keeps its MFMA pipe busy has room for about
// 1.6 VALU operations per 16x16x32 MFMA (measured: an MFMA holds the issue port for 9.5 of
// its 16.7 cycles, also against another wave's VALU operations).  Here a wave covers 64 rows,
// so a word feeds eight MFMAs, and the block's eight waves form 4 (N) x 2 (K) for INT4: the
// two K-waves of a tile take alternate 128-column groups and add their tiles in LDS, which
// keeps two waves per SIMD (one wave per SIMD with 64 x 96 tiles was slower: 63 against 50 us
// for gate/up at 128 rows, every scalar, LDS and wait instruction then takes an issue slot of
// the only wave).  BF16: 2 (M) x 4 (N) waves, 128 rows per block, so that the LM head's
// weights are read from HBM once per 128 rows instead of once per 64.
//
// Stages come by direct loads to LDS, a ring of two or three; the M0 register is set once per
// 4 KiB run (the instruction offset moves the LDS and the global address alike).  The
// activation fragments of the next k-step are read while the current one is multiplied, and
// one barrier per stage lies before its last k-step's MFMAs, so the reads behind it overlap
// them.
//
// INT4 d4096 layers: gate/up at 128 rows 55.5 -> 49.5 us; at 500 rows qkv 66 -> 59, wo 50 ->
// 40, gate/up 208 -> 200, down 110 -> 90 us.  LM head 32000 x 4096: 72 rows 112 -> 86, 128
// rows 98.6 -> 94.5, 500 rows 357 -> 329 us.
#include "gemm_tail.hpp"
#include "gemm_wide_rule.hpp"

namespace aarh {

static constexpr int GW_LDS = (int)MAX_DYN_LDS;
#define SCHED_FENCE __builtin_amdgcn_sched_barrier(0)

// LDS reads issued so far have returned.
__device__ __forceinline__ void wait_lds() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Four consecutive KiB (global and LDS) in one go: lds_dma16 with the instruction offset, which
// moves both addresses.
__device__ __forceinline__ void lds_dma4k(__amdgpu_buffer_rsrc_t r, const void* lds_dst, int voff, int soff) {
    const unsigned base = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds_dst);
    int saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %2, %3, %4 offen lds\n\t"
        "buffer_load_dwordx4 %2, %3, %4 offen offset:1024 lds\n\t"
        "buffer_load_dwordx4 %2, %3, %4 offen offset:2048 lds\n\t"
        "buffer_load_dwordx4 %2, %3, %4 offen offset:3072 lds\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "s"(base), "v"(voff), "s"(r), "s"(soff)
        : "memory");
}

// FMT INT4: one stage is a 128-column group of activations; the weight words (private to their
// wave) have a ring of their own.  FMT BF16: one stage is half a group of activations and
// weights.
template <int FMT, int CM, int CN, int WM, int WN, int WK>
struct GwCfg {
    static constexpr bool I4 = FMT == WF_INT4;
    static constexpr int NWV = WM * WN * WK;
    static constexpr int MC = WM * CM;                  // row chunks per block
    static constexpr int NT = WN * CN;                  // weight tiles per block
    static constexpr int SG = I4 ? 4 : 2;               // k-steps per stage
    static constexpr int AB = MC * SG * 2048;           // activation bytes of a K-wave's stage
    static constexpr int WB = I4 ? 0 : CN * SG * 1024;  // weight bytes of an N-wave's stage (BF16)
    static constexpr int STAGE = WK * AB + WN * WB;
    static constexpr int ZW = I4 ? 256 * ((CN + 3) / 4) : 0;
    static constexpr int WZ = I4 ? NWV * (CN * 1024 + ZW) : 0;  // INT4 weight + scale slot
    // stages: three where they fit, else two (INT4: two, and one weight slot)
    static constexpr int NS = 3 * STAGE + WZ <= GW_LDS ? 3 : 2;
    static_assert(!I4 || NS == 2, "the INT4 loop refills its one weight slot once a stage");
    static constexpr int LDS = NS * STAGE + WZ;
    static constexpr int LA = CM * SG * 2 / WN;             // activation loads per wave and stage
    static constexpr int LW = I4 ? CN + (CN + 3) / 4 : CN * SG / WM;  // weight (and scale) loads
    static constexpr int CPW = CM / WK;                     // chunks a wave keeps after the K reduction
    static_assert(CM * SG * 2 % WN == 0 && CM % WK == 0 && CN * SG % WM == 0, "pieces split over waves");
    static_assert(I4 ? WM == 1 : WK == 1, "INT4: K-waves share no weights; BF16: M-waves share them");
    static_assert(LDS <= GW_LDS, "ring exceeds LDS");
    static_assert((NS - 1) * (LA + LW) < 64, "vmcnt range");
    static_assert(NWV * 16 * CPW * (16 * CN + 4) * 4 <= LDS, "epilogue tile exceeds the ring");
    static_assert(NWV * (WK - 1) * CPW * CN * 1024 <= LDS, "K reduction exceeds the ring");
};

template <int FMT, int EPI, int CM, int CN, int WM, int WN, int WK>
__global__ void __launch_bounds__(WM * WN * WK * 64, 1) gemm_wide_kernel(GemvArgs a) {
    typedef GwCfg<FMT, CM, CN, WM, WN, WK> C;
    constexpr int NT = C::NT, MC = C::MC, CPW = C::CPW, NWV = C::NWV, NS = C::NS;
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    __shared__ float s_inv[MC * 16];
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int wk = wid / (WM * WN), wm = wid / WN % WM, wn = wid % WN;
    const int G = a.K >> 7, ntiles = a.N >> 4;
    const int NB = (ntiles + NT - 1) / NT, nchunks = (a.M + 15) >> 4;
    // (N-block, M-block): the M-blocks of one N-block run on one XCD (see gemm_kernel)
    const int bid = blockIdx.x;
    const int MBK = (int)gridDim.x / NB;
    const int full = NB / 8 * 8;
    int nb, mb;
    if (bid < full * MBK) {
        const int r = bid % (8 * MBK);
        mb = r / 8;
        nb = bid / (8 * MBK) * 8 + r % 8;
    } else {
        const int r = bid - full * MBK, w = NB - full;
        mb = r / w;
        nb = full + r % w;
    }
    const int n_it = (G + WK - 1) / WK;                    // group iterations of the block
    const int my_n = G > wk ? (G - wk + WK - 1) / WK : 0;  // of this wave
    const int nt0 = nb * NT + wn * CN;                       // the wave's first weight tile

    const __amdgpu_buffer_rsrc_t wr = coh_rsrc(a.w), fr = coh_rsrc(a.xf), zr = coh_rsrc(a.sz);
    auto grp = [&](int i) { return min(wk + WK * i, G - 1); };  // past the end: harmless repeats
    char* const a_lds = lds + wk * C::AB;
    char* const w_lds = lds + (C::I4 ? NS * C::STAGE + wid * (CN * 1024 + C::ZW)
                                                             : WK * C::AB + wn * C::WB);
    // stage h (SG k-steps each) into ring slot `slot`: the wave's share of the K-wave's chunks, and
    // (BF16) the wave's own weight tiles
    auto issue_stage = [&](int h, int slot) {
        const int g = grp(C::I4 ? h : h >> 1), half = C::I4 ? 0 : h & 1;
        char* base = a_lds + slot * C::STAGE;
        constexpr int RUNS = MC * C::SG / 2 / (WM * WN);  // 4 KiB runs per wave (two k-steps of a chunk)
        static_assert(RUNS >= 1, "a wave loads whole runs");
#pragma unroll
        for (int q = 0; q < RUNS; q++) {
            const int run = (wm * WN + wn) * RUNS + q, cc = run / (C::SG / 2), part = run % (C::SG / 2);
            const int mt = min(mb * MC + cc, nchunks - 1);
            lds_dma4k(fr, base + cc * C::SG * 2048 + part * 4096, lane * 16, (mt * G + g) * 8192 + (half + part) * 4096);
        }
        if constexpr (!C::I4) {
#pragma unroll
            for (int i = 0; i < C::LW; i++) {  // split over the M-waves
                const int pi = wm * C::LW + i, j = pi / C::SG, q = pi % C::SG;
                lds_dma16<true>(wr, w_lds + slot * C::STAGE + pi * 1024, lane * 16,
                             (int)(((unsigned)min(nt0 + j, ntiles - 1) * G + g) * 4096u + (half * 2 + q) * 1024u));
            }
        }
    };
    auto issue_w = [&](int i) {
        if constexpr (C::I4) {
            const int g = grp(i);
#pragma unroll
            for (int j = 0; j < CN; j++)
                lds_dma16<true>(wr, w_lds + j * 1024, lane * 16,
                             (int)(((unsigned)min(nt0 + j, ntiles - 1) * G + g) * 1024u));
#pragma unroll
            for (int q = 0; q < (CN + 3) / 4; q++) {
                const int zt = min(nt0 + min(4 * q + (lane >> 4), CN - 1), ntiles - 1);
                lds_dma4(zr, w_lds + CN * 1024 + q * 256, (int)(((unsigned)zt * G + g) * 64u + lr * 4u), 0);
            }
        }
    };

    // 1/rms of the block's rows from the producer's 16-column partial sums: wave w takes rows
    // w, w + NWV, ...  Up to K = 4096 (four partials per lane and row) they are loaded here,
    // ahead of the stages, and summed after the K loop.
    constexpr int RPW = MC * 16 / NWV;
    const bool norm_rows = a.norm_w != nullptr;
    const int nq = a.K >> 4;
    auto inv_rows = [&](const float (&ss)[RPW]) {
#pragma unroll
        for (int k = 0; k < RPW; k++) {
            float t = ss[k];
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) t += __shfl_xor(t, d, 64);
            if (lane == 0) s_inv[wid + NWV * k] = 1.0f / sqrtf(t / (float)a.K + a.eps);
        }
    };
    const bool inv_late = norm_rows && a.K <= 4096 && !(EPI == EPI_STORE && a.hidden_out);
    float iv[RPW][4];
    if (inv_late) {
#pragma unroll
        for (int k = 0; k < RPW; k++) {
            const int m = min(mb * MC * 16 + wid + NWV * k, a.M - 1);
#pragma unroll
            for (int u = 0; u < 4; u++) iv[k][u] = a.ssq_in[(size_t)m * a.ssq_ld + min(lane + 64 * u, nq - 1)];
        }
    }
    issue_w(0);
    issue_stage(0, 0);
    if constexpr (NS == 3) issue_stage(1, 1);
    issue_stage(NS - 1, NS - 1);
    if (norm_rows && !inv_late) {
        float ss[RPW];
#pragma unroll
        for (int k = 0; k < RPW; k++) ss[k] = 0.f;
        for (int q0 = lane; q0 < nq; q0 += 256)
#pragma unroll
            for (int k = 0; k < RPW; k++) {
                const int m = min(mb * MC * 16 + wid + NWV * k, a.M - 1);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const float v = a.ssq_in[(size_t)m * a.ssq_ld + min(q0 + 64 * u, nq - 1)];
                    if (q0 + 64 * u < nq) ss[k] += v;
                }
            }
        inv_rows(ss);
    }
    if (EPI == EPI_STORE && a.hidden_out) {
        // final normed hidden state (model.rs:579-585): the NB blocks of this M-block each write a
        // slice of columns of its rows
        __syncthreads();
        const int cw = ((a.K + NB - 1) / NB + 3) & ~3;
        const int k0 = nb * cw, kn = max(0, min(cw, a.K - k0));
        const int rows = min(MC * 16, a.M - mb * MC * 16);
        for (int idx = tid; idx < rows * (kn >> 2); idx += NWV * 64) {
            const int r = idx / (kn >> 2), k = k0 + 4 * (idx - r * (kn >> 2));
            const int m = mb * MC * 16 + r;
            const float4 v = *(const float4*)(a.x + row_off(a.xmap, m) + k);
            const float4 w = *(const float4*)(a.norm_w + k);
            const float si = s_inv[r];
            *(float4*)(a.hidden_out + (size_t)m * a.K + k) =
                make_float4(v.x * si * w.x, v.y * si * w.y, v.z * si * w.z, v.w * si * w.w);
        }
    }
    int pos[CPW][4];
    if (EPI == EPI_QKV)
#pragma unroll
        for (int c = 0; c < CPW; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int m = min((mb * MC + wm * CM + wk * CPW + c) * 16 + 4 * lg + i, a.M - 1);
                pos[c][i] = a.qkv.pos0[m / a.qkv.S] + m % a.qkv.S;
            }

    float4_t acc[CM][CN], ga[CM][CN];
#pragma unroll
    for (int c = 0; c < CM; c++)
#pragma unroll
        for (int j = 0; j < CN; j++) acc[c][j] = (float4_t){0.f, 0.f, 0.f, 0.f};

    u32x4_t ab[2][CM][2];              // activation fragments (hi, lo) of two k-steps
    u32x4_t wb[C::I4 ? 1 : 2][CN];     // INT4: words of the group, one per k-step; BF16: of two k-steps
    uint32_t szw[CN];
    const char* const a_ptr = lds + wk * C::AB + wm * CM * C::SG * 2048 + lg * 512 + lr * 16;
    const char* const w_ptr = w_lds;
    auto read_a = [&](int buf, int slot, int tt) {
        const char* base = a_ptr + slot * C::STAGE + tt * 2048;
#pragma unroll
        for (int c = 0; c < CM; c++) {
            ab[buf][c][0] = *(const u32x4_t*)(base + c * C::SG * 2048);
            ab[buf][c][1] = *(const u32x4_t*)(base + c * C::SG * 2048 + 256);
        }
        if constexpr (!C::I4)
#pragma unroll
            for (int j = 0; j < CN; j++)
                wb[buf][j] = ((const u32x4_t*)(w_ptr + slot * C::STAGE + (j * C::SG + tt) * 1024))[lane];
    };
    auto read_w = [&](u32x4_t (&w)[CN], uint32_t (&z)[CN]) {
#pragma unroll
        for (int j = 0; j < CN; j++) {
            w[j] = ((const u32x4_t*)(w_ptr + j * 1024))[lane];
            z[j] = ((const uint32_t*)(w_ptr + CN * 1024 + j * 64))[lr];
        }
    };
    half2_t zl2[CN], zh2[CN];
    float sc[CN];
    auto prep_z = [&]() {
#pragma unroll
        for (int j = 0; j < CN; j++) {
            sc[j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(szw[j] & 0xFFFFu));
            int4_zero_operands(__builtin_bit_cast(_Float16, (uint16_t)(szw[j] >> 16)), zl2[j], zh2[j]);
        }
    };
    // one k-step; t: its place in the group (INT4: the word, and the fresh group sum at t = 0)
    auto mfma_t = [&](int buf, int t) {
        const float4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < CN; j++) {
            if constexpr (C::I4) {
                const half8_t b = int4_b_operand(wb[0][j][t], zl2[j], zh2[j]);
#pragma unroll
                for (int c = 0; c < CM; c++)
                    ga[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, ab[buf][c][0]), b,
                                                                      t == 0 ? zero : ga[c][j], 0, 0, 0);
#pragma unroll
                for (int c = 0; c < CM; c++)
                    ga[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, ab[buf][c][1]), b,
                                                                      ga[c][j], 0, 0, 0);
            } else {
                const bf16x8_t b = __builtin_bit_cast(bf16x8_t, wb[buf][j]);
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int c = 0; c < CM; c++)
                        acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ab[buf][c][p]), b,
                                                                            acc[c][j], 0, 0, 0);
            }
        }
    };
    // the next stage (and its weights) has landed for every wave, and every wave has read the
    // stage before it (FIRST, LATER: loads issued after those)
    constexpr int FIRST = C::I4 ? (NS - 1) * C::LA + (NS - 2) * C::LW : (NS - 1) * (C::LA + C::LW);
    constexpr int LATER = (NS - 2) * (C::LA + C::LW);
    auto boundary = [&]() {
        wait_vmcnt<LATER>();
        __syncthreads();
    };
    auto next = [&](int x) { return x == NS - 1 ? 0 : x + 1; };

    wait_vmcnt<FIRST>();
    __syncthreads();
    read_a(0, 0, 0);
    if constexpr (C::I4) {
        read_w(wb[0], szw);
        prep_z();
        wait_lds();
        issue_w(1);
    }
    int sl = 0;
    if constexpr (C::I4) {
        for (int i = 0; i < n_it; i++) {
            u32x4_t wn_[CN];
            uint32_t zn_[CN];
            read_a(1, sl, 1);
            SCHED_FENCE;
            mfma_t(0, 0);
            SCHED_FENCE;
            read_a(0, sl, 2);
            SCHED_FENCE;
            mfma_t(1, 1);
            SCHED_FENCE;
            read_a(1, sl, 3);
            SCHED_FENCE;
            mfma_t(0, 2);
            SCHED_FENCE;
            boundary();
            issue_stage(i + NS, sl);
            sl = next(sl);
            SCHED_FENCE;
            read_a(0, sl, 0);
            read_w(wn_, zn_);
            SCHED_FENCE;
            mfma_t(1, 3);
            const bool on = i < my_n;
#pragma unroll
            for (int j = 0; j < CN; j++) {
                const float f = on ? sc[j] : 0.f;
#pragma unroll
                for (int c = 0; c < CM; c++) acc[c][j] += f * ga[c][j];
            }
            SCHED_FENCE;
#pragma unroll
            for (int j = 0; j < CN; j++) {
                wb[0][j] = wn_[j];
                szw[j] = zn_[j];
            }
            prep_z();
            wait_lds();  // the slot's words have been read
            issue_w(i + 2);
        }
    } else {
        for (int h = 0; h < 2 * n_it; h++) {
            read_a(1, sl, 1);
            SCHED_FENCE;
            mfma_t(0, 0);
            SCHED_FENCE;
            boundary();
            issue_stage(h + NS, sl);
            sl = next(sl);
            SCHED_FENCE;
            read_a(0, sl, 0);
            SCHED_FENCE;
            mfma_t(1, 0);
            SCHED_FENCE;
        }
    }
    wait_vmcnt<0>();
    if (inv_late) {
        float ss[RPW];
#pragma unroll
        for (int k = 0; k < RPW; k++) {
            ss[k] = 0.f;
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (lane + 64 * u < nq) ss[k] += iv[k][u];
        }
        inv_rows(ss);
    }
    __syncthreads();  // every wave's loads have landed and been read: the ring is free

    float4_t out[CPW][CN];
    if constexpr (WK > 1) {
        // the K-waves' partial tiles, added in K-wave order; wave wk keeps chunks wk CPW ..
        float4_t* red = (float4_t*)lds;
#pragma unroll
        for (int o = 0; o < WK; o++) {
            if (o == wk) continue;
            const int at = (((o * WN + wn) * (WK - 1) + (wk < o ? wk : wk - 1)) * CPW) * CN;
#pragma unroll
            for (int c = 0; c < CPW; c++)
#pragma unroll
                for (int j = 0; j < CN; j++) red[(at + c * CN + j) * 64 + lane] = acc[o * CPW + c][j];
        }
#pragma unroll
        for (int o = 0; o < WK; o++)
            if (o == wk)
#pragma unroll
                for (int c = 0; c < CPW; c++)
#pragma unroll
                    for (int j = 0; j < CN; j++) out[c][j] = acc[o * CPW + c][j];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < CPW; c++)
#pragma unroll
            for (int j = 0; j < CN; j++) {
                float4_t t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int o = 0; o < WK; o++) {
                    const int at = ((wid * (WK - 1) + (o < wk ? o : o - 1)) * CPW) * CN;
                    if (o == wk) t += out[c][j];
                    else t += red[(at + c * CN + j) * 64 + lane];
                }
                out[c][j] = t;
            }
        __syncthreads();
    } else {
#pragma unroll
        for (int c = 0; c < CPW; c++)
#pragma unroll
            for (int j = 0; j < CN; j++) out[c][j] = acc[c][j];
    }
    gemm_tail<FMT, EPI, CPW, CN, MC, NT>(a, 1, 0, mb, nb, NB, wm * CM + wk * CPW, wn * CN, out, pos, s_inv, lds, nullptr);
}

template <int FMT, int EPI, int CM, int CN, int WM, int WN, int WK>
static int launch_wide_cfg(const GemvArgs& a, hipStream_t stream) {
    typedef GwCfg<FMT, CM, CN, WM, WN, WK> C;
    static bool ready = false;
    if (!ready) {
        if (note_error(hipFuncSetAttribute((const void*)gemm_wide_kernel<FMT, EPI, CM, CN, WM, WN, WK>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS)))
            return 4;
        ready = true;
    }
    const int NB = (a.N / 16 + C::NT - 1) / C::NT, MB = ((a.M + 15) / 16 + C::MC - 1) / C::MC;
    (void)hipGetLastError();
    launch_timed(gemm_wide_kernel<FMT, EPI, CM, CN, WM, WN, WK>, dim3(NB * MB), dim3(C::NWV * 64), (uint32_t)C::LDS,
                 stream, a);
    return note_error(hipGetLastError()) ? 4 : 0;
}

bool gemm_wide_wins(const GemvArgs& a, int cus) {
    if (a.fmt == WF_BF16) return a.epi == EPI_STORE && wide_wins_head(a.N, a.M, cus);
    return a.fmt == WF_INT4 && wide_wins_int4(a.N, a.K, a.M, gemm_tuned(a), cus);
}

template <int EPI>
static int launch_wide_epi(const GemvArgs& a, int cus, hipStream_t stream) {
    if (a.fmt == WF_BF16) {
        if constexpr (EPI == EPI_STORE) return launch_wide_cfg<WF_BF16, EPI, 4, 2, 2, 4, 1>(a, stream);
        return 2;
    }
    if (wide_time(a.N, a.K, a.M, 3, cus) <= wide_time(a.N, a.K, a.M, 2, cus))
        return launch_wide_cfg<WF_INT4, EPI, 4, 3, 1, 4, 2>(a, stream);
    return launch_wide_cfg<WF_INT4, EPI, 4, 2, 1, 4, 2>(a, stream);
}

int launch_gemm_wide(const GemvArgs& a, int cus, hipStream_t stream) {
    switch (a.epi) {
        case EPI_STORE: return launch_wide_epi<EPI_STORE>(a, cus, stream);
        case EPI_RESID: return launch_wide_epi<EPI_RESID>(a, cus, stream);
        case EPI_SWIGLU: return launch_wide_epi<EPI_SWIGLU>(a, cus, stream);
        default: return launch_wide_epi<EPI_QKV>(a, cus, stream);
    }
}

}  // namespace aarh
