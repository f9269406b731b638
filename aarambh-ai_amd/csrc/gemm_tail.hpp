// Last part of the quantised GEMM kernels: split-K exchange and fused epilogue of
// the tiles a wave has accumulated (CPW chunks of 16 rows x TPW weight tiles in the
// MFMA accumulator layout).
#pragma once
#include "epilogue.hpp"

namespace aarh {

// s: the block's k-split of S; (mb, nb): its M-block (MC chunks) and N-block (NT tiles)
// of NB; the wave's tiles start at chunk wrow and tile wcol of the block.  pos: positions of
// the wave's rows (QKV).  s_inv: 1/rms of the block's rows (null norm_w: unused).  lds: a
// region of 16 CPW x (16 TPW + 4) floats per wave that no load writes any more.
template <int FMT, int EPI, int CPW, int TPW, int MC, int NT>
__device__ __forceinline__ void gemm_tail(const GemvArgs& a, int S, int s, int mb, int nb, int NB, int wrow, int wcol,
                                          float4_t (&acc)[CPW][TPW], const int (&pos)[CPW][4], const float* s_inv,
                                          char* lds, unsigned* s_flag) {
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int ntiles = a.N >> 4;
    const int row0 = (mb * MC + wrow) * 16, tile0 = nb * NT + wcol;
    // ---- epilogue inputs that do not depend on this kernel's products: loaded in the
    //      same round trip as the split-K partials (after the arrival, which waits for
    //      every outstanding access), or right away without a split ----
    int ntv[TPW];
#pragma unroll
    for (int j = 0; j < TPW; j++) ntv[j] = min(tile0 + j, ntiles - 1);
    // RESID: unit u = (row r, 8-column half s8 of a tile) of the wave's region; the old
    // residual and the next consumer's norm weights of every unit of the lane
    constexpr int TR = 16 * CPW, TLD = 16 * TPW + 4;
    constexpr int RU = TR * 2 * TPW, RI = (RU + 63) / 64;
    float rs[TPW];
    float xres[EPI == EPI_RESID ? RI : 1][8], nres[EPI == EPI_RESID ? RI : 1][8];
    float qcs[EPI == EPI_QKV ? TPW : 1][CPW][4], qsn[EPI == EPI_QKV ? TPW : 1][CPW][4];
    auto load_epi_inputs = [&]() {
        if (FMT == WF_INT8)
#pragma unroll
            for (int j = 0; j < TPW; j++) rs[j] = a.rscale[ntv[j] * 16 + lr];
        if (EPI == EPI_RESID) {
#pragma unroll
            for (int it = 0; it < RI; it++) {
                const int u = lane + 64 * it;
                const int r = u / (2 * TPW), s8 = u % (2 * TPW), m = row0 + r, nt = tile0 + (s8 >> 1);
                const int col = nt * 16 + (s8 & 1) * 8;
                const bool ok = u < RU && m < a.M && nt < ntiles;
                const float* xr = a.resid + (size_t)min(m, a.M - 1) * a.ldr + min(col, a.N - 8);
                if (ok && ((uintptr_t)xr & 15) == 0) {
                    const float4_t x0 = *(const float4_t*)xr, x1 = *(const float4_t*)(xr + 4);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        xres[it][e] = x0[e];
                        xres[it][4 + e] = x1[e];
                    }
                } else if (ok) {
#pragma unroll
                    for (int e = 0; e < 8; e++) xres[it][e] = xr[e];
                }
                if (ok && a.fo.buf && a.fo.norm_w)
#pragma unroll
                    for (int e = 0; e < 8; e++) nres[it][e] = a.fo.norm_w[col + e];
            }
        }
        // QKV: RoPE cos / sin of every (tile, row) of the lane
        if (EPI == EPI_QKV) {
            const int half = a.qkv.hd >> 1;
#pragma unroll
            for (int j = 0; j < TPW; j++) {
                const int rowq = ntv[j] * 16;
                const int d1 = 8 * ((rowq % a.qkv.hd) >> 4) + (lr & 7);
#pragma unroll
                for (int c = 0; c < CPW; c++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        qcs[j][c][i] = a.qkv.rope_cos[(size_t)pos[c][i] * half + d1];
                        qsn[j][c][i] = a.qkv.rope_sin[(size_t)pos[c][i] * half + d1];
                    }
            }
        }
    };
    if (S == 1) load_epi_inputs();

    if (S > 1) {
        // ---- split-K: partial tiles out, the last block of the (mb, nb) pair adds them in order ----
        const size_t unit = (size_t)mb * NB + nb;
        const __amdgpu_buffer_rsrc_t pr = coh_rsrc(a.gpart + unit * S * (MC * NT * 256));
#pragma unroll
        for (int c = 0; c < CPW; c++)
#pragma unroll
            for (int j = 0; j < TPW; j++) {
                const unsigned o = ((unsigned)(s * MC * NT + (wrow + c) * NT + wcol + j) * 64u + lane) * 16u;
                st4_coh(pr, o, acc[c][j]);
            }
        if (!arrive_last(a.gcnt + unit, (unsigned)S, s_flag)) return;
        load_epi_inputs();
        // the wave's CPW * TPW tiles x 4 splits in flight per round trip, added in split order
        const unsigned step = (unsigned)(MC * NT) * 1024u;
#pragma unroll
        for (int c = 0; c < CPW; c++)
#pragma unroll
            for (int j = 0; j < TPW; j++) acc[c][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < S; s0 += 4) {
            float4_t v[CPW][TPW][4];
#pragma unroll
            for (int c = 0; c < CPW; c++)
#pragma unroll
                for (int j = 0; j < TPW; j++) {
                    const unsigned o0 = ((unsigned)((wrow + c) * NT + wcol + j) * 64u + lane) * 16u;
#pragma unroll
                    for (int i = 0; i < 4; i++) v[c][j][i] = ld4_coh(pr, o0 + step * (unsigned)min(s0 + i, S - 1));
                }
#pragma unroll
            for (int c = 0; c < CPW; c++)
#pragma unroll
                for (int j = 0; j < TPW; j++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (s0 + i < S) acc[c][j] += v[c][j][i];
        }
    }

    // ---- epilogue in the MFMA layout: lane (lr, lg) of tile (c, j) holds rows
    //      4 lg + i of chunk c for weight row lr of tile j.  Its global inputs were
    //      loaded for all of the wave's tiles before the split-K exchange.
#pragma unroll
    for (int c = 0; c < CPW; c++)
#pragma unroll
        for (int j = 0; j < TPW; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float v = acc[c][j][i];
                if (a.norm_w) v *= s_inv[(wrow + c) * 16 + 4 * lg + i];
                if (FMT == WF_INT8) v *= rs[j];
                acc[c][j][i] = v;
            }

    // ---- the wave's tile goes through LDS (the stage ring is idle now) so that
    //      every global access is a 16-byte run of 4 (f32) or 8 (fragment)
    //      consecutive columns of one row ----
    float* wt = (float*)lds + wid * TR * TLD;
    if (EPI == EPI_QKV) {
        // a tile holds dims d = 8 jh + r (weight rows r < 8) and d + hd/2 (rows 8 + r) of one
        // head; RoPE (rope.rs:107-126) pairs lane lr with lane lr ^ 8, each keeps its own output
        const QkvEpi& e = a.qkv;
        const int QD = e.n_heads * e.hd, KD = e.n_kv * e.hd;
#pragma unroll
        for (int j = 0; j < TPW; j++) {
            const bool rot = ntv[j] * 16 < QD + KD;
#pragma unroll
            for (int c = 0; c < CPW; c++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float mine = acc[c][j][i], other = __shfl_xor(mine, 8, 64);
                    float y1 = lr < 8 ? mine : other, y2 = lr < 8 ? other : mine;
                    if (rot) {
#pragma clang fp contract(off)
                        const float r1 = y1 * qcs[j][c][i] - y2 * qsn[j][c][i];
                        const float r2 = y1 * qsn[j][c][i] + y2 * qcs[j][c][i];
                        y1 = r1;
                        y2 = r2;
                    }
                    wt[(16 * c + 4 * lg + i) * TLD + 16 * j + lr] = lr < 8 ? y1 : y2;
                }
            }
        }
    } else {
#pragma unroll
        for (int c = 0; c < CPW; c++)
#pragma unroll
            for (int j = 0; j < TPW; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) wt[(16 * c + 4 * lg + i) * TLD + 16 * j + lr] = acc[c][j][i];
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the wave's LDS writes are done
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    {
        if (EPI == EPI_SWIGLU) {
            // unit (row, tile): gate rows 0-7 and up rows 8-15 of the tile give h columns nt*8 .. +7
            for (int u = lane; u < TR * TPW; u += 64) {
                const int r = u / TPW, j = u % TPW, m = row0 + r, nt = tile0 + j;
                if (m >= a.M || nt >= ntiles) continue;
                const float4_t g0 = *(const float4_t*)(wt + r * TLD + 16 * j), g1 = *(const float4_t*)(wt + r * TLD + 16 * j + 4);
                const float4_t u0 = *(const float4_t*)(wt + r * TLD + 16 * j + 8), u1 = *(const float4_t*)(wt + r * TLD + 16 * j + 12);
                float h[8];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    h[e] = g0[e] / (1.0f + expf(-g0[e])) * u0[e];
                    h[4 + e] = g1[e] / (1.0f + expf(-g1[e])) * u1[e];
                }
                if (a.out) {  // f32 rows only for a consumer that reads them (f32 weights)
                    float* dst = a.out + row_off(a.omap, m) + nt * 8;
                    if (((uintptr_t)dst & 15) == 0) {
                        *(float4_t*)dst = (float4_t){h[0], h[1], h[2], h[3]};
                        *(float4_t*)(dst + 4) = (float4_t){h[4], h[5], h[6], h[7]};
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; e++) dst[e] = h[e];
                    }
                }
                if (a.fo.buf) {
                    if (a.fo.norm_w)
#pragma unroll
                        for (int e = 0; e < 8; e++) h[e] *= a.fo.norm_w[nt * 8 + e];
                    frag_put8_w(a.fo, m, nt * 8, h);
                }
            }
        } else if (EPI == EPI_STORE || EPI == EPI_RESID) {
            // unit (row, 8-column half of a tile); lanes 2q and 2q+1 hold the two halves of one tile row
#pragma unroll
            for (int it = 0; it < RI; it++) {  // RU is a multiple of 64 units, or 32
                const int u = lane + 64 * it;
                if (u >= RU) break;
                const int r = u / (2 * TPW), s8 = u % (2 * TPW), m = row0 + r, nt = tile0 + (s8 >> 1);
                const int col = nt * 16 + (s8 & 1) * 8;
                const bool ok = m < a.M && nt < ntiles;
                const float4_t v0 = *(const float4_t*)(wt + r * TLD + 8 * s8), v1 = *(const float4_t*)(wt + r * TLD + 8 * s8 + 4);
                float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                if (EPI == EPI_STORE) {
                    if (ok) {
                        float* dst = a.out + row_off(a.omap, m) + col;
                        if (((uintptr_t)dst & 15) == 0) {
                            *(float4_t*)dst = v0;
                            *(float4_t*)(dst + 4) = v1;
                        } else {
#pragma unroll
                            for (int e = 0; e < 8; e++) dst[e] = v[e];
                        }
                    }
                } else {
                    // x += y (old x loaded before the split-K exchange); the new x as fragments
                    // for the next consumer and its 16-column sums of squares
                    float sq = 0.f;
                    if (ok) {
                        float* xr = a.resid + (size_t)m * a.ldr + col;
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            v[e] += xres[it][e];
                            sq += v[e] * v[e];
                        }
                        if (((uintptr_t)xr & 15) == 0) {
                            *(float4_t*)xr = (float4_t){v[0], v[1], v[2], v[3]};
                            *(float4_t*)(xr + 4) = (float4_t){v[4], v[5], v[6], v[7]};
                        } else {
#pragma unroll
                            for (int e = 0; e < 8; e++) xr[e] = v[e];
                        }
                        if (a.fo.buf) {
                            if (a.fo.norm_w)
#pragma unroll
                                for (int e = 0; e < 8; e++) v[e] *= nres[it][e];
                            frag_put8_w(a.fo, m, col, v);
                        }
                    }
                    sq += __shfl_xor(sq, 1, 64);
                    if (a.fo.ssq && ok && (s8 & 1) == 0) a.fo.ssq[(size_t)m * a.fo.ssq_ld + nt] = sq;
                }
            }
        } else if (EPI == EPI_QKV) {
            // unit (row, tile): dims 8 jh .. +7 and 8 jh + hd/2 .. +7 of one head
            const QkvEpi& e = a.qkv;
            const int hd = e.hd, half = hd >> 1;
            const int QD = e.n_heads * hd, KD = e.n_kv * hd;
            for (int u = lane; u < TR * TPW; u += 64) {
                const int r = u / TPW, j = u % TPW, m = row0 + r, nt = tile0 + j;
                if (m >= a.M || nt >= ntiles) continue;
                const int rowq = nt * 16, head = rowq / hd, d0 = 8 * ((rowq % hd) >> 4);
                float* dst;
                if (rowq < QD) dst = e.q_out + (size_t)m * QD + head * hd;
                else if (rowq < QD + KD) dst = e.kv_out + (size_t)m * 2 * KD + (head - e.n_heads) * hd;
                else dst = e.kv_out + (size_t)m * 2 * KD + KD + (head - e.n_heads - e.n_kv) * hd;
                const float* src = wt + r * TLD + 16 * j;
                float* p1 = dst + d0;
                float* p2 = dst + d0 + half;
                if ((((uintptr_t)p1 | (uintptr_t)p2) & 15) == 0) {
                    *(float4_t*)p1 = *(const float4_t*)src;
                    *(float4_t*)(p1 + 4) = *(const float4_t*)(src + 4);
                    *(float4_t*)p2 = *(const float4_t*)(src + 8);
                    *(float4_t*)(p2 + 4) = *(const float4_t*)(src + 12);
                } else {
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        p1[q] = src[q];
                        p2[q] = src[8 + q];
                    }
                }
            }
        }
    }
}

}  // namespace aarh
