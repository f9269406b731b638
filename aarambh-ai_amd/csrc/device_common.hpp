// Device-side helpers shared by the gfx950 kernels of libaarambh_hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "exact_f32.hpp"

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef short bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));

#define WAVE 64

// Build-defined synthetic generator (same formula as the test oracle):
// splitmix64 counter hash -> Box-Muller in f64.
__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__device__ __forceinline__ float synth_normal(uint64_t seed, uint32_t stream, uint64_t index) {
    uint64_t base = splitmix64(seed ^ ((uint64_t)stream * 0xD1B54A32D192ED03ull));
    uint64_t h = splitmix64(base + index);
    double u1 = ((double)(h >> 40) + 1.0) * (1.0 / 16777216.0);
    double u2 = (double)((h >> 16) & 0xFFFFFFull) * (1.0 / 16777216.0);
    return (float)(sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2));
}

// f32::total_cmp ordering key: larger key == larger value, NaN above +inf.
__device__ __forceinline__ int32_t total_key(float f) {
    int32_t i = __float_as_int(f);
    return i ^ (int32_t)(((uint32_t)(i >> 31)) >> 1);
}

// exp rounded to nearest f32: evaluate in f64 and round once.  This matches a
// correctly rounded libm expf except in the rare cases where the host libm
// itself misrounds; those show up as flagged near-ties, never silently.
__device__ __forceinline__ float expf_rn(float x) { return (float)exp((double)x); }

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
    uint32_t x = __float_as_uint(f);
    if ((x & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((x >> 16) | 0x40u);
    x += 0x7FFFu + ((x >> 16) & 1u);
    return (uint16_t)(x >> 16);
}

// ---------------------------------------------------------------------------
// rand 0.8 StdRng (ChaCha12, rand_chacha 0.3.1) seeded by seed_from_u64
// (rand_core 0.6.4): keystream word n of sequence seed, evaluated on device.
// ---------------------------------------------------------------------------
// Byte offset, inside one 16-row x 128-column weight tile, of byte b of lane l's
// share (TILE_BYTES / 64 bytes: row l % 16, columns 32 * (l / 16) .. +32 of the
// group).  The share is cut into 16-byte chunks and chunk q of every lane sits in
// the q-th KiB of the tile, lanes in order: a 16-byte load per lane reads one
// contiguous KiB.  INT4 shares are a single chunk.
__host__ __device__ __forceinline__ int tile_byte(int lane, int b) { return ((b >> 4) << 10) + lane * 16 + (b & 15); }

__device__ __forceinline__ uint32_t rotl32(uint32_t v, int n) { return (v << n) | (v >> (32 - n)); }

__device__ inline void rng_key_from_seed(uint64_t state, uint32_t key[8]) {
    const uint64_t mul = 6364136223846793005ull, inc = 11634580027462260723ull;
    for (int i = 0; i < 8; i++) {
        state = state * mul + inc;
        uint32_t xs = (uint32_t)(((state >> 18) ^ state) >> 27);
        uint32_t rot = (uint32_t)(state >> 59);
        key[i] = (xs >> rot) | (xs << ((32 - rot) & 31));
    }
}

#define CHACHA_QR(a, b, c, d)                                                                      \
    a += b; d ^= a; d = rotl32(d, 16);                                                             \
    c += d; b ^= c; b = rotl32(b, 12);                                                             \
    a += b; d ^= a; d = rotl32(d, 8);                                                              \
    c += d; b ^= c; b = rotl32(b, 7);

__device__ inline uint32_t rng_word(const uint32_t key[8], uint64_t word) {
    uint32_t in[16] = {0x61707865u, 0x3320646eu, 0x79622d32u, 0x6b206574u,
                       key[0], key[1], key[2], key[3], key[4], key[5], key[6], key[7],
                       (uint32_t)(word >> 4), (uint32_t)(word >> 36), 0u, 0u};
    uint32_t x[16];
#pragma unroll
    for (int i = 0; i < 16; i++) x[i] = in[i];
    for (int r = 0; r < 12; r += 2) {
        CHACHA_QR(x[0], x[4], x[8], x[12]);
        CHACHA_QR(x[1], x[5], x[9], x[13]);
        CHACHA_QR(x[2], x[6], x[10], x[14]);
        CHACHA_QR(x[3], x[7], x[11], x[15]);
        CHACHA_QR(x[0], x[5], x[10], x[15]);
        CHACHA_QR(x[1], x[6], x[11], x[12]);
        CHACHA_QR(x[2], x[7], x[8], x[13]);
        CHACHA_QR(x[3], x[4], x[9], x[14]);
    }
    uint32_t idx = (uint32_t)(word & 15);
    uint32_t out = 0;
#pragma unroll
    for (int i = 0; i < 16; i++)
        if ((uint32_t)i == idx) out = x[i] + in[i];
    return out;
}

// rand 0.8 Standard f32: (next_u32 >> 8) * 2^-24.
__device__ inline float rng_f32(const uint32_t key[8], uint64_t word) {
    return (float)(rng_word(key, word) >> 8) * (1.0f / 16777216.0f);
}

// ---------------------------------------------------------------------------
// Cross-workgroup hand-off without L2 flushes.
//
// A device-scope fence on gfx950 writes back the whole XCD L2 (buffer_wbl2),
// which costs microseconds per workgroup.  Data that one workgroup hands to
// another inside a kernel (split-K partials, row statistics) is instead written
// and read with agent-scope relaxed atomics, which compile to sc1 (coherent,
// L2-bypassing) stores/loads; the writer waits for its stores to complete
// (s_waitcnt vmcnt(0)) before it signals arrival on the counter.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void st_coh(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_coh_i32(int32_t* p, int32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_coh(const float* p) {
    return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int32_t ld_coh_i32(const int32_t* p) {
    return __hip_atomic_load(const_cast<int32_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// All of this thread's memory operations have completed.
// 16-byte agent-coherent global access through a raw buffer resource (cache policy
// sc1: the access is performed at device scope, past the per-XCD L2 state), for
// partial results handed between workgroups of one launch.  Offsets in bytes.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t coh_rsrc(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ float4_t ld4_coh(__amdgpu_buffer_rsrc_t r, unsigned byte_off) {
    return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r, (int)byte_off, 0, 16));
}
__device__ __forceinline__ float2_t ld2_coh(__amdgpu_buffer_rsrc_t r, unsigned byte_off) {
    return __builtin_bit_cast(float2_t, __builtin_amdgcn_raw_buffer_load_b64(r, (int)byte_off, 0, 16));
}
__device__ __forceinline__ void st4_coh(__amdgpu_buffer_rsrc_t r, unsigned byte_off, float4_t v) {
    typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), r, (int)byte_off, 0, 16);
}
__device__ __forceinline__ void wait_mem() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
// Called by every thread of the workgroup after its coherent stores; returns
// true in the workgroup that arrives last (which also re-arms the counter).
__device__ __forceinline__ bool arrive_last(unsigned* counter, unsigned expected, unsigned* s_flag) {
    wait_mem();
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned prev = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bool last = prev == expected - 1u;
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *s_flag = last ? 1u : 0u;
    }
    __syncthreads();
    bool last = *s_flag != 0u;
    wait_mem();
    return last;
}

// ---------------------------------------------------------------------------
// Wave-level primitives
// ---------------------------------------------------------------------------
__device__ __forceinline__ int wave_excl_scan_i32(int v) {
    const int lane = threadIdx.x & 63;
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        int t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    return incl - v;
}

__device__ __forceinline__ float wave_max_f32(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    return v;
}

__device__ __forceinline__ float wave_sum_f32(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

// ---------------------------------------------------------------------------
// Exact sequential f32 summation on one wave.
//
// Continues s_k = fl(s_{k-1} + v[k]) over v[0..n) for v[k] >= 0 from the running
// sum st.s, bit-identical to a scalar left-to-right f32 loop (the reference's
// iter().sum::<f32>() and the running cumulative of sample_from_probs), so a long
// vector can be summed in pieces.  With u >= 0 it also records the first k with
// u <= s_k (inverse CDF, `draw <= cumulative`), as gbase + k.
//
// Method: while s stays inside one binade [2^e, 2^(e+1)), every partial sum
// is an integer multiple of ulp(s), and fl(s + x) = s + ulp * RNE(x / ulp)
// unless x / ulp has fraction exactly 1/2 (a tie, decided by parity).  So the
// wave turns 512 elements (8 consecutive ones per lane, held in registers) into integer
// increments and scans them over the lanes.  The lanes before the first one that
// leaves the binade, holds a tie or reaches u are taken at once; that lane's 8 elements
// are added one after another with real f32 adds.  The lanes after it keep their
// increments if the sum is still in the binade, and are turned again otherwise.
// ---------------------------------------------------------------------------
struct SeqScan {
    float s;         // running sum
    int cross;       // first global index k with u <= s_k; -1 while none
    float s_at;      // s_cross
    float s_before;  // s_{cross-1} (0 before the first element)
};

__device__ __forceinline__ SeqScan seq_scan_init() {
    SeqScan st;
    st.s = 0.0f;
    st.cross = -1;
    st.s_at = 0.0f;
    st.s_before = 0.0f;
    return st;
}

// Inclusive prefix sum over the 64 lanes with DPP row shifts and row broadcasts
// (register-to-register, no LDS round trip per step).
__device__ __forceinline__ int wave_incl_scan_dpp(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2, 3
    return v;
}
__device__ __forceinline__ float readlane_f32(float x, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

constexpr int SCAN_WIN = 512;  // elements per window: 8 per lane

// LDS pointers as such: the scans are functions of their own (one copy of their code for all
// callers), where a plain pointer would be read through the flat path.
typedef __attribute__((address_space(3))) const float lds_cfloat;
typedef __attribute__((address_space(3))) const float4_t lds_cfloat4;

// The lane's 8 elements of the window v[0..n), n <= SCAN_WIN (0 past the end).
__device__ __forceinline__ void scan_load(lds_cfloat* v, int n, float (&x)[8]) {
    const int base = 8 * (threadIdx.x & 63);
    if (base + 8 <= n) {
        const float4_t a = *(lds_cfloat4*)(v + base), b = *(lds_cfloat4*)(v + base + 4);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            x[k] = a[k];
            x[4 + k] = b[k];
        }
    } else {
#pragma unroll
        for (int k = 0; k < 8; k++) x[k] = base + k < n ? v[base + k] : 0.0f;
    }
}

// Sums of at least 2^-103 (biased exponent 24 up) are scanned by increments as they are: the
// scale 2^sft is then a normal f32 and x * 2^sft is exact or far above 2^24.
constexpr int SCAN_MIN_EB = 24;
__device__ __forceinline__ float scan_pow2(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// Sum of the lane's increments RNE(x / ulp), ulp = 2^-sft.  `special`: an element is a tie or
// not a finite value in [0, 2^24) ulps (its bit pattern, read as unsigned, is at or above
// that of 2^24: also negative values and NaN), or the sum leaves any binade.
__device__ __forceinline__ int scan_increments(const float (&x)[8], int sft, bool& special) {
    const float scale = scan_pow2(sft);
    int lsum = 0;
    float dmax = 0.0f;
    uint32_t bmax = 0u;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const float c = x[k] * scale;
        const float rr = __builtin_rintf(c);
        dmax = fmaxf(dmax, fabsf(c - rr));
        bmax = max(bmax, __float_as_uint(c));
        lsum += (int)rr;
    }
    special = bmax >= 0x4B800000u || dmax == 0.5f || lsum >= 16777216;
    return special ? 0 : lsum;
}

// Continues st over one window (x from scan_load, n elements, the first one index gbase).
__device__ __forceinline__ void scan_window(const float (&x)[8], int n, float u, int gbase, SeqScan& st) {
    const int lane = threadIdx.x & 63;
    const int lanes = (n + 7) >> 3;
    float s = st.s;
    int from = 0;  // first lane not yet added
    // the elements of lane `stop`, one f32 add each
    auto add_lane = [&](int stop) __attribute__((always_inline)) {
        if (u >= 0.0f && st.cross < 0) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float before = s;
                s = before + readlane_f32(x[k], stop);
                if (st.cross < 0 && u <= s && 8 * stop + k < n) {
                    st.cross = gbase + 8 * stop + k;
                    st.s_at = s;
                    st.s_before = before;
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) s += readlane_f32(x[k], stop);
        }
        from = stop + 1;
    };
    while (from < lanes) {
        const uint32_t bits = (uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(s));
        if (bits >= 0x7F800000u) {  // infinite or NaN
            add_lane(from);
            continue;
        }
        // Zero and subnormal sums count in the ulps of the first binade, 2^-149, where every
        // increment is exact.  Sums below 2^-103 are counted with all values times 2^64 (exact,
        // or infinite and so special).  At low temperatures a row's sum stays there until its
        // first sizable term.  With the lanes of such windows added one by one, 28 sequences x 9
        // rows of 32 000 logits took 419 us at temperature 0.1 and 2512 us at 0.02 (one lane is
        // 0.4 us); counted this way 167 and 174 us, as at ordinary temperatures.
        const int eb = max((int)(bits >> 23), 1);
        const bool tiny = eb < SCAN_MIN_EB;
        const float up = tiny ? 0x1p64f : 1.0f, down = tiny ? 0x1p-64f : 1.0f;
        const int sft = 150 - eb - (tiny ? 64 : 0);          // x / ulp(s) == x * up * 2^sft
        const float ulp = scan_pow2(-sft);                   // ulp(s) / down
        auto ulps = [&](uint32_t b) { return (int)(b - ((uint32_t)(eb - 1) << 23)); };
        int base = ulps(bits);                               // s / ulp(s), less the increments of lanes < from
        float y[8];
#pragma unroll
        for (int k = 0; k < 8; k++) y[k] = x[k] * up;
        bool special;
        int lsum = scan_increments(y, sft, special);
        if (lane < from) lsum = 0;
        const int incl = wave_incl_scan_dpp(lsum);
        for (;;) {
            const int end = base + incl;
            const bool halt = special || end >= 16777216 ||
                              (u >= 0.0f && st.cross < 0 && u <= (float)end * ulp * down);
            const unsigned long long m = __ballot(halt && lane >= from);
            const int stop = m ? __ffsll((long long)m) - 1 : 64;
            s = (float)(stop == 64 ? __builtin_amdgcn_readlane(end, 63)
                                   : __builtin_amdgcn_readlane(end - lsum, stop)) * ulp * down;
            if (stop >= lanes) {
                from = lanes;
                break;
            }
            add_lane(stop);
            const uint32_t nb = (uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(s));
            if (from >= lanes || max((int)(nb >> 23), 1) != eb) break;
            base = ulps(nb) - __builtin_amdgcn_readlane(incl, stop);
        }
    }
    st.s = s;
}

// Continues st over v[0..n) in LDS; lane l of isum / wexp: the integer sum of window l in ulps
// (-1: unusable) and the binade it holds for, predicted by the caller.
__device__ __noinline__ static SeqScan seq_scan_chunk(lds_cfloat* v, int n, float u, int gbase, SeqScan st, int isum, int wexp) {
    n = __builtin_amdgcn_readfirstlane(n);
    gbase = __builtin_amdgcn_readfirstlane(gbase);
#pragma unroll 1
    for (int w = 0; w * SCAN_WIN < n; w++) {
        const int add = w < 64 ? __builtin_amdgcn_readlane(isum, w) : -1;
        const int eb = w < 64 ? __builtin_amdgcn_readlane(wexp, w) : 0;
        const uint32_t bits = (uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(st.s));
        if (add >= 0 && (int)(bits >> 23) == eb) {
            const int end = (int)((bits & 0x7FFFFFu) | 0x800000u) + add;
            const float s1 = (float)end * scan_pow2(eb - 150);
            if (end < 16777216 && !(u >= 0.0f && st.cross < 0 && u <= s1)) {
                st.s = s1;
                continue;
            }
        }
        float x[8];
        scan_load(v + w * SCAN_WIN, min(SCAN_WIN, n - w * SCAN_WIN), x);
        scan_window(x, min(SCAN_WIN, n - w * SCAN_WIN), u, gbase + w * SCAN_WIN, st);
    }
    return st;
}

// One 1 KiB wave load straight into LDS: lane l's 16 bytes at rsrc + voff +
// soff land at LDS address lds_base + 16 l (buffer_load_dwordx4 ... lds, base in
// M0).  Written as inline asm so the compiler does not see an LDS write it would
// guard with a conservative vmcnt(0) before every LDS read: the kernel counts
// these loads itself.  M0 is restored before the statement ends.  NT marks the load
// non-temporal (data read once: a stream of weights or cache blocks).
template <bool NT = false>
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t r, const void* lds_dst, int voff, int soff) {
    const unsigned base = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds_dst);
    int saved;
    if constexpr (NT)
        asm volatile(
            "s_mov_b32 %0, m0\n\t"
            "s_mov_b32 m0, %1\n\t"
            "s_nop 0\n\t"
            "buffer_load_dwordx4 %2, %3, %4 offen nt lds\n\t"
            "s_mov_b32 m0, %0"
            : "=&s"(saved)
            : "s"(base), "v"(voff), "s"(r), "s"(soff)
            : "memory");
    else
        asm volatile(
            "s_mov_b32 %0, m0\n\t"
            "s_mov_b32 m0, %1\n\t"
            "s_nop 0\n\t"
            "buffer_load_dwordx4 %2, %3, %4 offen lds\n\t"
            "s_mov_b32 m0, %0"
            : "=&s"(saved)
            : "s"(base), "v"(voff), "s"(r), "s"(soff)
            : "memory");
}

// One 256-byte wave load into LDS: lane l's 4 bytes land at lds_dst + 4 l.
template <bool NT = false>
__device__ __forceinline__ void lds_dma4(__amdgpu_buffer_rsrc_t r, const void* lds_dst, int voff, int soff) {
    const unsigned base = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds_dst);
    int saved;
    if constexpr (NT)
        asm volatile(
            "s_mov_b32 %0, m0\n\t"
            "s_mov_b32 m0, %1\n\t"
            "s_nop 0\n\t"
            "buffer_load_dword %2, %3, %4 offen nt lds\n\t"
            "s_mov_b32 m0, %0"
            : "=&s"(saved)
            : "s"(base), "v"(voff), "s"(r), "s"(soff)
            : "memory");
    else
        asm volatile(
            "s_mov_b32 %0, m0\n\t"
            "s_mov_b32 m0, %1\n\t"
            "s_nop 0\n\t"
            "buffer_load_dword %2, %3, %4 offen lds\n\t"
            "s_mov_b32 m0, %0"
            : "=&s"(saved)
            : "s"(base), "v"(voff), "s"(r), "s"(soff)
            : "memory");
}

// s_waitcnt vmcnt(n) (gfx9 encoding: vmcnt[3:0] | vmcnt[5:4] << 14), other counters unconstrained.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}
