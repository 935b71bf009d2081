// exl3_gemm_rd.hip -- the register-decode GEMM: EXL3 linears of a decode batch (up to 128 rows) on gfx950.
//
// y = had_out(fp16(had_in(x) . W), svh) for rows that one tile holds (32 R rows, R = 1 to 4): two
// launches, the input transform (launch_had, in fragment order) and this kernel.
//
// What bounds it.  Every weight is decoded once, ~4 vector instructions a weight whatever the rows (the
// GEMV's bound too), and the matrix cores' share grows with R: 141 / 156 / 152 / 160 vector (R = 1 to 4; the
// whole kernel's count over its loop's steps) and 4 R matrix instructions (32 cycles each) per 32 k x 64
// columns and wave.  The two hardly overlap: counted at gate/up 5120 -> 2 x 17408, 4 bpw, vector issue takes
// 70 / 65 / 54 / 49 % of a busy CU's cycles and the matrix cores 16 / 27 / 35 / 40 % at 32 / 64 / 96 / 128 rows,
// 86 to 92 % together.  The 256-row prefill kernel pays its LDS
// round trip of the weights and a barrier per 64 k for rows that are not there (gate 5120 -> 17408: 1.1
// us a step, 60 us, at 64 rows as at 256).  Here a wave keeps what it decodes:
//   * a lane's q-block is a 32x32x16 MFMA's B operand as it stands (lane bit 5: k-tile, bits 4..0:
//     n-tile and q; the q-block's column halves and row halves select the MFMA), so the weights go
//     from the decoder to the matrix cores without LDS and without another wave;
//   * the input comes in the fragment order of that MFMA (frag_offset): contiguous 16-byte loads
//     straight into operand registers, no LDS, no barrier in the loop;
//   * a workgroup is 8 waves, 2 column halves x 4 K groups of one 128-column tile, two waves a SIMD
//     (up to 256 registers), one workgroup a CU; the K groups meet in LDS once per tile.
// The work is cut along K over the CUs (rd_plan); pieces of one tile meet through fp32 partial tiles
// and a counter, as the prefill's split tiles do (device-scope stores, vmcnt(0), one relaxed add,
// device-scope loads by the last contributor, sums in workgroup order).
// Measured (4 bpw, graphs of 16 launches over cold weights, transform included; before: the faster of
// GEMV and prefill GEMM): gate/up 5120 -> 2 x 17408 at 16 / 32 / 64 / 96 / 128 rows 42 / 57 / 89 / 113 /
// 118 -> 38 / 40 / 53 / 65 / 79 us; gate 29 / 41 / 60 / 65 / 67 -> 25 / 26 / 34 / 43 / 51; 5120 -> 5120 19 /
// 26 / 34 / 36 / 37 -> 15 / 16 / 21 / 25 / 28; at 32 rows such a step takes a SIMD 0.37 us (gate/up's 85 of
// them against 5120 -> 5120's 20), the other ~9 us are the transform's launch, the first loads and the completion.
#include "exl3_gemm_rd.h"

#include <algorithm>

using namespace exl3;

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct RdGroup {
    const uint16_t* xf;         // rotated input in fragment order (M * K halves, below 2^31 bytes)
    const uint32_t* trellis;
    const uint16_t* svh;
    uint16_t* y;                // first output column of the group (rows ldy apart)
    int n;                      // columns
    int w0, G;                  // its workgroups: grid [w0, w0 + G)
    int tile0;                  // its first completion counter
    UDiv d_u, d_g;              // divisions by its units and its workgroups
};

struct RdArgs {
    int64_t ldy;
    int M, K, groups;
    UDiv d_upt;                 // division by the units of a tile
    f32x4* part;                // [2 grid][RD partial tile]: slot 2 b of workgroup b's first segment, 2 b + 1 of its last
    uint32_t part_bytes;
    uint32_t* counters;         // one per tile, zero between calls
    RdGroup g[EXL3_MAX_GROUPS];
};

// LDS barrier without a wait for global loads in flight
__device__ __forceinline__ void rd_barrier()
{
    __builtin_amdgcn_sched_barrier(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);                // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_sched_barrier(0);
}

// quad VQ of an MFMA accumulator (by value: element accesses through a pointer can end in scratch)
template <int VQ>
__device__ __forceinline__ f32x4 quad(f32x16 v)
{
    return __builtin_shufflevector(v, v, 4 * VQ, 4 * VQ + 1, 4 * VQ + 2, 4 * VQ + 3);
}

// f(0) .. f(N - 1) with constant indices (a loop that is not unrolled would leave its array in scratch)
template <int N, class F>
__device__ __forceinline__ void repeat(F&& f)
{
    static_for(std::make_integer_sequence<int, N>{}, f);
}

constexpr int C_ROW = 136;                             // LDS row (halves) of a tile's fp16 C

// ---- a workgroup's range of units, the exchange of partial tiles and the output transform ----------
// A tile is 32 R rows x 128 columns; its fp32 accumulators move as 16 R "slots" of 64 lanes x 16
// bytes in register order: slot ((2 wc + h) R + i) 4 + vq holds, in lane l and element e, row
// 32 i + 8 vq + 4 (l >> 5) + e, column 64 wc + 8 h + 16 ((l >> 3) & 3) + (l & 7).  A thread holds NQ
// consecutive slots' quads from slot0 on.
template <int BITS, int R, int NQ, int WAVES>
struct RdWork {
    const RdArgs& a;
    RdGroup gg;
    int b, wave, lane, t;
    int UPT;                                           // units (256 k) of a tile
    uint32_t U, G, w;                                  // units and workgroups of the group, this workgroup
    int ulo, uhi, tile_first, slot0;
    __amdgpu_buffer_rsrc_t prs;

    __device__ __forceinline__ RdWork(const RdArgs& args) : a(args)
    {
        b = blockIdx.x;
        t = threadIdx.x;
        wave = __builtin_amdgcn_readfirstlane(t >> 6);
        lane = t & 63;
        int gi = 0;
        if (a.groups > 1 && b >= a.g[1].w0) gi = 1;
        if (a.groups > 2 && b >= a.g[2].w0) gi = 2;
        if (a.groups > 3 && b >= a.g[3].w0) gi = 3;
        gg = gi == 0 ? a.g[0] : gi == 1 ? a.g[1] : gi == 2 ? a.g[2] : a.g[3];
        UPT = a.K / 256;
        U = (uint32_t) (gg.n / 128) * (uint32_t) UPT;
        G = (uint32_t) gg.G;
        w = (uint32_t) (b - gg.w0);
        ulo = lo_of(w);
        uhi = lo_of(w + 1);
        tile_first = tile_of(ulo);
        prs = __builtin_amdgcn_make_buffer_rsrc(a.part, 0, (int) a.part_bytes, RAW_BUFFER_FLAGS);
    }
    // workgroup c owns units [lo_of(c), lo_of(c + 1))
    __device__ __forceinline__ int lo_of(uint32_t c) const { return (int) gg.d_g.div(U * c); }
    __device__ __forceinline__ int tile_of(int u) const { return (int) a.d_upt.div((uint32_t) u); }
    // a tile's first and last contributor
    __device__ __forceinline__ int first_wg(int tile) const { return (int) gg.d_u.div((uint32_t) (tile * UPT + 1) * G - 1u); }
    __device__ __forceinline__ int last_wg(int tile) const { return (int) gg.d_u.div((uint32_t) (tile * UPT + UPT) * G - 1u); }
    __device__ __forceinline__ uint32_t quad_off(int i) const { return (uint32_t) (slot0 + i) * 1024u + (uint32_t) lane * 16u; }

    // partial slot sl (16 R KB each): 2 b for workgroup b's first segment, 2 b + 1 for its last
    template <int N>
    __device__ __forceinline__ void store_part(uint32_t sl, const f32x4 (&sum)[N], int i0 = 0) const
    {
        repeat<N>([&](auto I) __attribute__((always_inline)) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum[I]), prs, quad_off(i0 + I), sl * (uint32_t) (16 * R * 1024), SC1);
        });
    }
    // a tile's partials (N quads of the thread from i0 on) summed in workgroup order, the loads of several
    // contributors in flight
    template <int N>
    __device__ __forceinline__ void gather(int tile, int wf, int wl, f32x4 (&tot)[N], int i0 = 0) const
    {
        // the first contributor's partial is its last segment's unless its range starts with the tile
        const uint32_t s0 = 2u * (uint32_t) (gg.w0 + wf) + (lo_of((uint32_t) wf) == tile * UPT ? 0u : 1u);
        repeat<N>([&](auto I) __attribute__((always_inline)) { tot[I] = f32x4{0.f, 0.f, 0.f, 0.f}; });
        constexpr int B = N <= 4 ? 4 : 2;
        for (int c0 = wf; c0 <= wl; c0 += B) {
            f32x4 v[B][N];
            repeat<B>([&](auto K_) __attribute__((always_inline)) {
                const int c = min(c0 + (int) K_, wl);
                const uint32_t sl = c == wf ? s0 : 2u * (uint32_t) (gg.w0 + c);
                repeat<N>([&](auto I) __attribute__((always_inline)) {
                    v[K_][I] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(prs, quad_off(i0 + I), sl * (uint32_t) (16 * R * 1024), SC1));
                });
            });
            repeat<B>([&](auto K_) __attribute__((always_inline)) {
                const float live = c0 + (int) K_ <= wl ? 1.f : 0.f;
                repeat<N>([&](auto I) __attribute__((always_inline)) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) tot[I][e] = live != 0.f ? tot[I][e] + v[K_][I][e] : tot[I][e];
                });
            });
        }
    }
    // fp16 C of a tile into LDS, [32 R][C_ROW] halves
    __device__ __forceinline__ void put_c(uint16_t* ct, const f32x4 (&sum)[NQ]) const
    {
        repeat<NQ>([&](auto I) __attribute__((always_inline)) {
            const int sl = slot0 + I, vq = sl & 3, rt = (sl >> 2) % R, ch = (sl >> 2) / R;
            const int col = (ch >> 1) * 64 + (ch & 1) * 8 + ((lane >> 3) & 3) * 16 + (lane & 7);
            const int row = 32 * rt + 8 * vq + 4 * (lane >> 5);
#pragma unroll
            for (int e = 0; e < 4; ++e) ct[(row + e) * C_ROW + col] = f16_bits((f16) sum[I][e]);
        });
    }
    // y = fp16(fp16(Had128(C)) * svh) of a tile's C, 16-byte write-through stores.  Up to 64 rows the
    // float64 butterflies of the fused GEMV (exact sums), above them the prefill's float32 sums on the
    // matrix cores (had128_mfma16: the values of exl3_had_r_128_f32).
    static constexpr bool EXACT = R <= 2;
    __device__ __forceinline__ void emit(const uint16_t* ct, int tile, int first_wave, int n_waves) const
    {
        const int col0 = tile * 128, jr = lane & 15, gq = lane >> 4;
        const __amdgpu_buffer_rsrc_t svs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(gg.svh), 0, 0x7FFFFFFF, RAW_BUFFER_FLAGS);
        const __amdgpu_buffer_rsrc_t ysrc = __builtin_amdgcn_make_buffer_rsrc(gg.y, 0, 0x7FFFFFFF, RAW_BUFFER_FLAGS);
        auto sv_at = [&](int c) __attribute__((always_inline)) {
            return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(svs, (uint32_t) ((col0 + c) * 2), 0, SC1));
        };
        auto store = [&](int r, int c, u32x4 v) __attribute__((always_inline)) {
            if (r < a.M)
                __builtin_amdgcn_raw_buffer_store_b128(v, ysrc, (uint32_t) (((int64_t) r * a.ldy + col0 + c) * 2), 0, SC1);
        };
        if constexpr (EXACT) {                                    // 16 lanes a row, 4 rows a wave
            const u32x4 sv = sv_at(8 * jr);
            for (int r4 = 4 * (wave - first_wave); r4 < a.M; r4 += 4 * n_waves) {
                const u32x4 c = *reinterpret_cast<const u32x4*>(ct + (r4 + gq) * C_ROW + 8 * jr);
                store(r4 + gq, 8 * jr, had128_x8<double>(c, u32x4{0u, 0u, 0u, 0u}, false, sv, true, r_scale<double>()));
            }
        } else {                                                  // 16 rows a wave
            u32x4 sv[4];
            repeat<4>([&](auto P) __attribute__((always_inline)) { sv[P] = sv_at(32 * P + 8 * gq); });
            const HadMfmaA HA = had_mfma_a();
            for (int rg = wave - first_wave; 16 * rg < a.M; rg += n_waves) {
                const int r = rg * 16 + jr;
                u32x4 xb[4];
                repeat<4>([&](auto S) __attribute__((always_inline)) { xb[S] = *reinterpret_cast<const u32x4*>(ct + r * C_ROW + 32 * S + 8 * gq); });
                had128_mfma16(HA, xb, r_scale<float>(), true, sv, [&](int p, u32x4 v) __attribute__((always_inline)) { store(r, 32 * p + 8 * gq, v); });
            }
        }
    }
    // a whole tile of this workgroup (lds: free, all waves past a barrier)
    __device__ __forceinline__ void whole_tile(char* lds, int tile, const f32x4 (&sum)[NQ]) const
    {
        uint16_t* const ct = reinterpret_cast<uint16_t*>(lds);
        put_c(ct, sum);
        rd_barrier();
        emit(ct, tile, 0, WAVES);
    }
    // count this workgroup into the tiles it left partials of: the first segment's (pend; p_others other
    // contributors) and the last one's (e_part); done: it was the last contributor
    __device__ __forceinline__ void count(int* s_last, bool pend, bool e_part, int tp, int te, int p_others, int e_others, bool& p_done,
                                          bool& e_done) const
    {
        __builtin_amdgcn_s_waitcnt(0x0F70);                       // vmcnt(0): the partials have landed
        rd_barrier();
        if (t < 2 && (t == 0 ? pend : e_part)) {
            uint32_t* const c = &a.counters[gg.tile0 + (t == 0 ? tp : te)];
            const uint32_t prev = __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool last = prev == (uint32_t) (t == 0 ? p_others : e_others);
            s_last[t] = last;
            if (last) __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        rd_barrier();
        p_done = pend && s_last[0];
        if (e_part) e_done = s_last[1];
    }
    // the end of the range: `sum` is the last segment's, `pend` says that the first segment's partial
    // was stored (its count was put off to here); the last contributor of a tile finishes it
    __device__ __forceinline__ void end_range(char* lds, int* s_last, bool pend, f32x4 (&sum)[NQ]) const
    {
        const int te = tile_of(uhi - 1);
        const int ef = first_wg(te), el = last_wg(te), pf = first_wg(tile_first), pl = last_wg(tile_first);
        const bool e_part = ef != el;
        if (e_part) store_part(2u * (uint32_t) b + (te != tile_first ? 1u : 0u), sum);
        bool p_done = false, e_done = !e_part;
        if (e_part || pend) {
            count(s_last, pend, e_part, tile_first, te, pl - pf, el - ef, p_done, e_done);
        } else {
            rd_barrier();                                         // the sums are read
        }
        uint16_t* const ct = reinterpret_cast<uint16_t*>(lds);
        if (!p_done && !e_done) return;                           // uniform
        if (p_done) {
            f32x4 tot[NQ];
            gather(tile_first, pf, pl, tot);
            put_c(ct, tot);
        }
        if (e_done) {
            if (e_part) gather(te, ef, el, sum);
            put_c(ct + 32 * R * C_ROW, sum);
        }
        rd_barrier();
        // two tiles: half of the waves each
        if (p_done && e_done) {
            const bool second = wave >= WAVES / 2;
            emit(ct + (second ? 32 * R * C_ROW : 0), second ? te : tile_first, second ? WAVES / 2 : 0, WAVES / 2);
        } else {
            emit(ct + (e_done ? 32 * R * C_ROW : 0), e_done ? te : tile_first, 0, WAVES);
        }
    }
};

// a load cursor over the units of a range; it stops at the range's last unit (reloaded, never used)
struct RdCur {
    int u, ku, tile;
    __device__ __forceinline__ void advance(int uhi, int UPT)
    {
        if (u + 1 >= uhi) return;
        ++u;
        if (++ku < UPT) return;
        ku = 0;
        ++tile;
    }
};

template <int R>
struct Rd {
    static constexpr int DA = R == 1 ? 4 : R <= 3 ? 2 : 1;                    // sub-steps of input fragments in flight
    static constexpr int SLOTS = 16 * R;
    static constexpr int LDS = (R == 1 ? 8 : R == 2 ? 4 : 2) * SLOTS * 1024;
};

template <int BITS, int CB, int R>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) gemm_rd_kernel(RdArgs a)
{
    using P_ = Rd<R>;
    constexpr int DA = P_::DA, NQ = 2 * R;
    extern __shared__ __align__(16) char lds[];
    __shared__ int s_last[2];
    RdWork<BITS, R, NQ, 8> W(a);
    const int lane = W.lane, wave = W.wave, wc = wave & 1, kg = wave >> 1;
    W.slot0 = wave * NQ;
    const int M = a.M, K = a.K, nt_total = W.gg.n / 16, UPT = W.UPT, ulo = W.ulo, uhi = W.uhi;

    const __amdgpu_buffer_rsrc_t trs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(W.gg.trellis), 0, (int) ((uint32_t) (K / 16) * (uint32_t) nt_total * 32u * BITS), RAW_BUFFER_FLAGS);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(W.gg.xf), 0, (int) ((uint32_t) M * (uint32_t) K * 2u), RAW_BUFFER_FLAGS);

    // trellis: lane (b5: k-tile of the pair, b4 b3: n-tile of the wave's four, b2..0: q-block)
    const int q = lane & 7;
    const uint32_t tile_w = (uint32_t) ((2 * kg + (lane >> 5)) * nt_total + 4 * wc + ((lane >> 3) & 3)) * (8 * BITS);
    const uint32_t off_main = (tile_w + q * BITS) * 4u;
    const uint32_t off_prev = (tile_w + (q == 0 ? 8 * BITS - 1 : q * BITS - 1)) * 4u;
    const uint32_t step_d = (uint32_t) nt_total * 8u * 32u * BITS, step_u = 2 * step_d;

    RdCur cw{ulo, ulo - W.tile_first * UPT, W.tile_first}, ca = cw;
    auto woff_of = [&]() __attribute__((always_inline)) { return (uint32_t) cw.tile * (8u * 32u * BITS) + (uint32_t) cw.ku * step_u; };
    uint32_t woff = woff_of();
    uint32_t Wr[4][BITS + 1];
    auto fetch_w = [&](auto S) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
        load_qblock_buf<BITS>(trs, off_main, off_prev, woff + (s & 1) * step_d, Wr[s]);
        if (s & 1) {
            cw.advance(uhi, UPT);
            woff = woff_of();
        }
    };

    // input fragments: row tile T (32 rows) holds, for each 32-k slice and 8-row half rh of a
    // k-tile, lanes (k-tile, row) of 16 bytes; the last tile holds its live rows only
    uint32_t aoff[R], arow[R];
    repeat<R>([&](auto I) __attribute__((always_inline)) {
        const uint32_t rows = (uint32_t) min(32, M - 32 * (int) I);
        arow[I] = rows;
        aoff[I] = I * 64u * (uint32_t) K + ((uint32_t) (lane >> 5) * rows + min((uint32_t) (lane & 31), rows - 1u)) * 16u;
    });
    f16x8 A[DA][R][2];
    auto fetch_a1 = [&](auto S, auto I, auto RH) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value, i = decltype(I)::value, rh = decltype(RH)::value;
        const uint32_t kk = (uint32_t) (ca.ku * 8 + (s & 1) * 4 + kg);
        A[s % DA][i][rh] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(xrs, aoff[i], (kk * 64u + rh * 32u) * arow[i], 0));
    };
    auto a_done = [&](auto S) __attribute__((always_inline)) {       // every fragment of sub-step S requested
        if constexpr (decltype(S)::value & 1) ca.advance(uhi, UPT);
    };

    f32x16 acc[R][2];
    auto clear = [&]() __attribute__((always_inline)) {
        repeat<R>([&](auto I) __attribute__((always_inline)) { acc[I][0] = acc[I][1] = f32x16{}; });
    };
    clear();

    // sub-step S (ring slot): decode this wave's 32 k x 64 columns, multiply, refill
    auto sub = [&](auto S, bool refill) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
        uint32_t P[16];
        decode_qblock<BITS, CB>(Wr[s], P);
        static_for(std::make_integer_sequence<int, 2>{}, [&](auto RH) __attribute__((always_inline)) {
            constexpr int rh = decltype(RH)::value;
            const u32x4 B0 = {P[rh], P[4 + rh], P[8 + rh], P[12 + rh]};
            const u32x4 B1 = {P[2 + rh], P[6 + rh], P[10 + rh], P[14 + rh]};
            static_for(std::make_integer_sequence<int, R>{}, [&](auto I) __attribute__((always_inline)) {
                constexpr int i = decltype(I)::value;
                acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[s % DA][i][rh], __builtin_bit_cast(f16x8, B0), acc[i][0], 0, 0, 0);
                acc[i][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[s % DA][i][rh], __builtin_bit_cast(f16x8, B1), acc[i][1], 0, 0, 0);
                fetch_a1(std::integral_constant<int, s + DA>{}, I, RH);
            });
        });
        a_done(std::integral_constant<int, s + DA>{});
        // after the fragments: loads return in order, and the fragments (cached) would wait for it
        __builtin_amdgcn_sched_barrier(0);
        if (refill) fetch_w(S);
    };

    // this wave's accumulators into K group `region`'s slots in LDS
    auto put = [&](int region) __attribute__((always_inline)) {
        repeat<8 * R>([&](auto I) __attribute__((always_inline)) {      // (h, i, vq)
            constexpr int h = decltype(I)::value / (4 * R), i = decltype(I)::value / 4 % R, vq = decltype(I)::value & 3;
            *reinterpret_cast<f32x4*>(lds + (region * P_::SLOTS + wc * 8 * R + I) * 1024 + lane * 16) = quad<vq>(acc[i][h]);
        });
    };
    // the sum of the four K groups from `region` on
    auto ksum = [&](int region, f32x4 (&sum)[NQ]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const char* p = lds + region * P_::SLOTS * 1024 + W.quad_off(i);
            f32x4 v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const f32x4*>(p + k * P_::SLOTS * 1024);
            sum[i] = (v[0] + v[2]) + (v[1] + v[3]);
        }
    };
    // more than 64 rows: two regions; groups 2 and 3 join 0 and 1 first (all waves past a barrier)
    auto ksum2 = [&](f32x4 (&sum)[NQ]) __attribute__((always_inline)) {
        if (kg >= 2) put(kg - 2);
        rd_barrier();
        if (kg < 2)
            repeat<8 * R>([&](auto I) __attribute__((always_inline)) {
                constexpr int h = decltype(I)::value / (4 * R), i = decltype(I)::value / 4 % R, vq = decltype(I)::value & 3;
                const f32x4 v = *reinterpret_cast<const f32x4*>(lds + (kg * P_::SLOTS + wc * 8 * R + I) * 1024 + lane * 16);
                acc[i][h][4 * vq] += v[0];
                acc[i][h][4 * vq + 1] += v[1];
                acc[i][h][4 * vq + 2] += v[2];
                acc[i][h][4 * vq + 3] += v[3];
            });
        rd_barrier();
        if (kg < 2) put(kg);
        rd_barrier();
        repeat<NQ>([&](auto I) __attribute__((always_inline)) {
            const char* p = lds + W.quad_off(I);
            sum[I] = *reinterpret_cast<const f32x4*>(p) + *reinterpret_cast<const f32x4*>(p + P_::SLOTS * 1024);
        });
    };
    // The first segment when it does not end the range: its K groups' sums wait in LDS (pend 1) or its
    // partial is stored (pend 2); no wave waits for another until the end of the range.
    int pend = 0;
    auto flush_pend = [&]() __attribute__((always_inline)) {       // on entry: all waves past a barrier
        f32x4 sum[NQ];
        ksum(0, sum);
        W.store_part(2u * (uint32_t) W.b, sum);
        pend = 2;
    };
    auto mid = [&](int u) __attribute__((always_inline)) {          // a tile ends inside the range
        const int tile = W.tile_of(u - 1);
        if (R <= 2 && W.first_wg(tile) != W.last_wg(tile)) {
            put(kg);
            pend = 1;
        } else if (R > 2) {
            f32x4 sum[NQ];
            rd_barrier();
            ksum2(sum);
            if (W.first_wg(tile) != W.last_wg(tile)) {
                W.store_part(2u * (uint32_t) W.b, sum);
                pend = 2;
            } else {
                rd_barrier();
                W.whole_tile(lds, tile, sum);
            }
        } else {                                                   // a whole tile
            rd_barrier();
            if (pend == 1) {
                flush_pend();
                rd_barrier();
            }
            put(kg);
            rd_barrier();
            f32x4 sum[NQ];
            ksum(0, sum);
            rd_barrier();
            W.whole_tile(lds, tile, sum);
        }
        clear();
    };

    static_for(std::make_integer_sequence<int, 4>{}, fetch_w);
    static_for(std::make_integer_sequence<int, DA>{}, [&](auto S) __attribute__((always_inline)) {
        static_for(std::make_integer_sequence<int, R>{}, [&](auto I) __attribute__((always_inline)) {
            fetch_a1(S, I, std::integral_constant<int, 0>{});
            fetch_a1(S, I, std::integral_constant<int, 1>{});
        });
        a_done(S);
    });
    int left = UPT - (ulo - W.tile_first * UPT);                  // units of the current tile still to come
    int u = ulo;
    auto unit_end = [&]() __attribute__((always_inline)) {
        ++u;
        if (--left == 0 && u < uhi) {
            mid(u);
            left = UPT;
        }
    };
    while (u + 2 <= uhi) {
        sub(std::integral_constant<int, 0>{}, true);
        sub(std::integral_constant<int, 1>{}, true);
        unit_end();
        sub(std::integral_constant<int, 2>{}, true);
        sub(std::integral_constant<int, 3>{}, true);
        unit_end();
    }
    if (u < uhi) {
        sub(std::integral_constant<int, 0>{}, false);
        sub(std::integral_constant<int, 1>{}, false);
    }
    f32x4 sum[NQ];
    if constexpr (R == 1) {
        put(4 + kg);                                              // apart from a pending segment's sums
        rd_barrier();
        if (pend == 1) flush_pend();
        ksum(4, sum);
    } else if constexpr (R == 2) {
        rd_barrier();
        if (pend == 1) {
            flush_pend();
            rd_barrier();
        }
        put(kg);
        rd_barrier();
        ksum(0, sum);
    } else {
        rd_barrier();
        ksum2(sum);
    }
    W.end_range(lds, s_last, pend != 0, sum);
}

}  // namespace

namespace {

constexpr int RD_CUS = 256;                    // MI355X compute units: one workgroup each

template <int LDS>
int launch_rd_k(void (*kern)(RdArgs), bool& attr_set, int threads, const RdArgs& a, int grid, hipStream_t s)
{
    if (!attr_set) {                         // dynamic LDS above 64 KB must be enabled per kernel
        if (hipFuncSetAttribute((const void*) kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess)
            return EXL3_ELAUNCH;
        attr_set = true;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), LDS, s, a);
    return hipGetLastError() == hipSuccess ? EXL3_OK : EXL3_ELAUNCH;
}

template <int BITS, int CB, int R>
int launch_rd_t(const RdArgs& a, int grid, hipStream_t s)
{
    static bool attr_set = false;
    return launch_rd_k<Rd<R>::LDS>(gemm_rd_kernel<BITS, CB, R>, attr_set, 512, a, grid, s);
}

template <int BITS, int CB>
int launch_rd_r(int R, const RdArgs& a, int grid, hipStream_t s)
{
    switch (R) {
        case 1: return launch_rd_t<BITS, CB, 1>(a, grid, s);
        case 2: return launch_rd_t<BITS, CB, 2>(a, grid, s);
        case 3: return launch_rd_t<BITS, CB, 3>(a, grid, s);
        default: return launch_rd_t<BITS, CB, 4>(a, grid, s);
    }
}

template <int BITS>
int launch_rd_cb(int cb, int R, const RdArgs& a, int grid, hipStream_t s)
{
    switch (cb) {
        case 0: return launch_rd_r<BITS, 0>(R, a, grid, s);
        case 1: return launch_rd_r<BITS, 1>(R, a, grid, s);
        default: return launch_rd_r<BITS, 2>(R, a, grid, s);
    }
}

}  // namespace

// Workgroups of a launch.  A group's units are shared evenly by its G workgroups, [floor(U c / G),
// floor(U (c + 1) / G)).  With G = tiles x s every tile is cut into s pieces of its own and no
// workgroup works on two tiles: worth more than an even share, because a workgroup with the end of
// one tile and the start of another stores, counts and may finish two (12288 columns, 96 tiles x 20
// units: 192 workgroups of half a tile 20.5 / 26.1 / 30.2 / 34.4 us at 16 / 64 / 96 / 128 rows, 256
// workgroups of 7.5 units 21.2 / 30.8 / 37.3 / 44.8).  Fewer pieces leave CUs idle, more of them make
// the last one of a tile read more partials.  The choice is the least of this cost, in units, fitted
// to 16 shapes at 8 to 128 rows: the longest piece, 0.55 a piece of a tile, 0.02 a workgroup, and 4.5
// where pieces cross tiles (256 workgroups, the only way with more tiles than CUs: gate / up 5120 ->
// 2 x 17408; one 17408 takes it too, 24.9 / 34.3 / 51.0 us at 16 / 64 / 128 rows against 29.5 / 37.7 /
// 53.8 for 136 whole tiles).
RdPlan rd_plan(int M, int K, const int* widths, int groups)
{
    RdPlan p{};
    // K below 2048 (at most 7 units a tile) stays with the prefill kernel.  Below 1024 that never splits a
    // tile, so its launches are bitwise equal to reconstruct + hgemm and between grouped and single calls,
    // which cut tiles are not; from 1024 to 2047 this kernel was not measured
    if (M < 1 || M > RD_MAX_ROWS || K % 256 || K < 2048) return p;
    // the rotated input of a group is read through a raw buffer with 32-bit byte offsets
    if ((uint64_t) M * (uint64_t) K * 2 >= (1ull << 31)) return p;
    const int64_t upt = K / 256;
    int64_t tiles = 0;
    for (int i = 0; i < groups; ++i) {
        p.tile0[i] = (int) tiles;
        tiles += widths[i] / 128;
    }
    if (tiles > RD_MAX_TILES || tiles * upt * RD_CUS >= (1ll << 31)) return p;
    p.R = (M + 31) / 32;
    int pieces = 0;                                               // 0: an even share, pieces cross tiles
    double best = (double) (tiles * upt) / RD_CUS + 0.55 * (1.0 + (double) RD_CUS / tiles) + 0.02 * RD_CUS + 4.5;
    for (int64_t s = 1; s <= upt && tiles * s <= RD_CUS; ++s) {
        const double c = (double) ((upt + s - 1) / s) + 0.55 * s + 0.02 * (double) (tiles * s);
        if (c < best || (pieces == 0 && tiles * upt < RD_CUS)) {
            best = c;
            pieces = (int) s;
        }
    }
    int64_t given = 0;
    for (int i = 0; i < groups; ++i) {
        const int64_t t = widths[i] / 128;
        p.G[i] = (int) (pieces ? t * pieces : std::max<int64_t>(1, RD_CUS * t / tiles));
        given += p.G[i];
    }
    while (!pieces && given < RD_CUS) {                           // the rest to the groups with the most units per workgroup
        int m = 0;
        for (int i = 1; i < groups; ++i)
            if ((int64_t) widths[i] * p.G[m] > (int64_t) widths[m] * p.G[i]) m = i;
        ++p.G[m];
        ++given;
    }
    for (int i = 0; i < groups; ++i) {
        p.w0[i] = p.grid;
        p.grid += p.G[i];
    }
    p.part_bytes = (size_t) p.grid * 2 * 16 * p.R * 1024;
    p.use = true;
    return p;
}

// The kernel's unit split of a plan against brute force: 0, the number of mismatches, or -1 for a
// shape the plan does not serve.
static int rd_check(int M, int K, const int* widths, int groups)
{
    const RdPlan p = rd_plan(M, K, widths, groups);
    if (!p.use) return -1;
    int bad = 0, w0 = 0, tile0 = 0;
    const int upt = K / 256;
    for (int i = 0; i < groups; ++i) {
        const int tiles = widths[i] / 128;
        const uint32_t U = (uint32_t) (tiles * upt), G = (uint32_t) p.G[i];
        const UDiv du = UDiv::of(U), dg = UDiv::of(G), dt = UDiv::of((uint32_t) upt);
        bad += p.w0[i] != w0 || p.tile0[i] != tile0 || G < 1 || G > U;
        w0 += p.G[i];
        tile0 += tiles;
        uint32_t lo = 0;
        for (uint32_t c = 0; c < G; ++c) {                        // ranges: consecutive, none empty, all units
            const uint32_t a = dg.div(U * c), b = dg.div(U * (c + 1));
            bad += a != lo || b <= a || a != (uint64_t) U * c / G;
            for (uint32_t u = a; u < b; ++u) {                    // every owner found by the contributors' formulas
                const uint32_t t = dt.div(u);
                const uint32_t wf = du.div((t * upt + 1) * G - 1u), wl = du.div((t * upt + upt) * G - 1u);
                bad += t != u / upt || c < wf || c > wl;
                if (u == t * upt) bad += c != wf;
                if (u == t * upt + upt - 1) bad += c != wl;
            }
            lo = b;
        }
        bad += lo != U;
    }
    bad += w0 != p.grid || p.part_bytes != (size_t) p.grid * 2 * 16 * p.R * 1024;
    return bad;
}

extern "C" int exl3_gemm_rd_check(int m, int k, const int* widths, int groups)
{
    if (!widths || groups < 1 || groups > EXL3_MAX_GROUPS) return -1;
    for (int i = 0; i < groups; ++i)
        if (widths[i] < 128 || widths[i] % 128) return -1;
    return rd_check(m, k, widths, groups);
}

int launch_gemm_rd(const RdPlan& pl, int bits, int cb, const uint16_t* const* xf, const void* const* trellis, uint16_t* const* y,
                   int64_t ldy, const uint16_t* const* svh, const int* widths, int groups, int M, int K, void* part, uint32_t* counters,
                   hipStream_t s)
{
    RdArgs a{};
    a.ldy = ldy;
    a.M = M;
    a.K = K;
    a.groups = groups;
    a.counters = counters;
    a.part = (f32x4*) part;
    a.part_bytes = (uint32_t) pl.part_bytes;
    for (int i = 0; i < groups; ++i)
        a.g[i] = {xf[i], (const uint32_t*) trellis[i], svh[i], y[i], widths[i], pl.w0[i], pl.G[i], pl.tile0[i],
                  UDiv::of((uint32_t) (widths[i] / 128 * (K / 256))), UDiv::of((uint32_t) pl.G[i])};
    a.d_upt = UDiv::of((uint32_t) (K / 256));
    switch (bits) {
        case 1: return launch_rd_cb<1>(cb, pl.R, a, pl.grid, s);
        case 2: return launch_rd_cb<2>(cb, pl.R, a, pl.grid, s);
        case 3: return launch_rd_cb<3>(cb, pl.R, a, pl.grid, s);
        case 4: return launch_rd_cb<4>(cb, pl.R, a, pl.grid, s);
        case 5: return launch_rd_cb<5>(cb, pl.R, a, pl.grid, s);
        case 6: return launch_rd_cb<6>(cb, pl.R, a, pl.grid, s);
        case 7: return launch_rd_cb<7>(cb, pl.R, a, pl.grid, s);
        default: return launch_rd_cb<8>(cb, pl.R, a, pl.grid, s);
    }
}
