// gemm.hip -- the prompt's projections C[M][N] = A[M][K] W[N][K]^T on CDNA4
// fp16 MFMA (gfx950), with the neighbouring row-wise work in the epilogue:
// the residual add, SwiGLU of gate and up columns, or the q/k/v split with
// RoPE.
//
// At 2048 rows the matrix cores are busy 47 % of a gate/up product (11264 x
// 2048, at 1.9 GHz), 38 % of down, 27 % of o and 23 % of QKV (tiles that leave CUs
// idle), LDS 24 / 29 / 20 / 12 % without bank conflicts; few rows wait for weights
// that no cache holds, and small tiles for the L2 -> CU path (64 bytes a clock and
// CU), so the tile is chosen per shape (gemm_pick).
//
// Tile BN x BM (weight rows x prompt rows), K in steps of 64.  A stage holds
// the step's BN rows of W and BM rows of A, 128 bytes a row, filled by
// global_load_lds_dwordx4 (8 rows an instruction); 16-byte chunk c of row r
// sits at c ^ (r / 2 % 8), so that the 16-byte operand reads of 16 neighbouring
// rows, two rows to a 256-byte bank line, hit distinct banks.  NS stages form a
// ring.
//
// v_mfma_f32_32x32x16_f16 with W as the A operand: lane (h, col) = (l / 32,
// l % 32) ends with rows 8u + 4h .. +4 (u = 0..3) of W for prompt row col, four
// consecutive output columns each (8-byte stores).  Paired epilogues order the
// tile's rows in groups of 32 that alternate first and second member (gate /
// up rows, RoPE dims d / d + D/2), so both members of a pair meet in one lane.
//
// A step is four quarters of 16 of K; a wave reads the next quarter's operands
// while the MFMAs of this one run, and over the first three quarters loads step
// t+NS-1 into the slot of step t-1.  Before the last quarter's MFMAs it waits
// for its own loads of step t+1 and meets the workgroup (every wave is done
// reading step t, and step t+1 has landed), then reads the first quarter of
// step t+1.
#include "kvhp_internal.h"

#include <algorithm>

namespace kvhp {

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) f16 lds_f16;
typedef __attribute__((address_space(3))) void lds_void;

enum GemmEpi : int { kGemmResidual = 0, kGemmSwiglu = 1, kGemmQKV = 2, kGemmF32 = 3 };

struct GemmArgs {
    const f16* A;          // [M][K]
    const f16* W;          // [N][K] (SwiGLU: gate rows, then up rows)
    f16* out;              // residual [M][N] (in place), SwiGLU [M][N/2], QKV q [M][Hq*D]
    float* out32;          // fp32 [M][N], of each K range its own
    int M, N, K;           // N: weight rows
    int n_tiles, m_tiles;
    int k_steps;           // steps of a K range (blockIdx.y)
    int Hq, Hkv, D;
    const float2* rope;    // [M][D/2] (cos, sin)
    f16* k;                // [M][Hkv*D]
    f16* v;
};

// global_load_lds_dwordx4: lane l's 16 bytes land at lds_base + 16 l.  Inline
// asm, so that only the explicit vmcnt waits order it against the LDS reads.
__device__ __forceinline__ void dma16s(const f16* sbase, uint32_t voff, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(lds_base), "v"(voff), "s"(sbase) : "memory", "m0");
}

template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// This wave's LDS reads complete, then the workgroup meets; loads stay in flight.
__device__ __forceinline__ void stage_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ float r16(float v) { return static_cast<float>(static_cast<f16>(v)); }

// silu(g) u for a gate rounded to fp16: the bits of g / (1 + expf(-g)) u at all
// 65536 gates, on half the instructions.  The exponent -g log2(e) is an exact
// product (g has 11 bits, the constant's head 13) plus the rest of the constant;
// the quotient is a reciprocal's product and one residual step, in sixteenths so
// that no reciprocal is subnormal.  Where the residual is zero, or NaN (infinite
// gates and exponentials), the product stands.  v_exp_f32 of the rounded product
// and v_rcp_f32 are up to 61 units of 2^-24 off, expf and this 2.4; a 2048-id
// prompt of the 22-layer 2048 / 5632 model takes 1.1-1.4 % longer than with those
// two (5500 against 5440 us), and 2.7 % with expf and the IEEE division.
__device__ __forceinline__ float silu_mul(float g, float u) {
    constexpr float hi = -1.442626953125f, lo = static_cast<float>(-1.4426950408889634 - hi);
    const float gc = __builtin_amdgcn_fmed3f(g, -200.f, 200.f);   // exp(-g) infinite or 0 beyond
    const float t = gc * hi, n = rintf(t);
    const float e = ldexpf(fast_exp2(fmaf(gc, lo, t - n)), static_cast<int>(n));
    const float d = fmaf(e, 0.0625f, 0.0625f), g16 = g * 0.0625f;
    const float r = __builtin_amdgcn_rcpf(d), q = g16 * r, res = fmaf(-d, q, g16);
    return (__builtin_islessgreater(res, 0.f) ? fmaf(res, r, q) : q) * u;
}

template <int BN, int BM, int BK, int WN, int WM, int NS, int EPI>
__global__ void __launch_bounds__(WN * WM * kWave)
gemm_kernel(const GemmArgs a) {
    constexpr int NW = WN * WM;
    constexpr int TN = BN / WN / 32, TM = BM / WM / 32;   // 32x32 tiles of a wave
    constexpr int ROWS = BN + BM;
    constexpr int CPR = BK / 8;                           // 16-byte chunks per staged row
    constexpr int RPI = kWave / CPR;                      // rows per load instruction
    constexpr int LPT = ROWS / RPI / NW;                  // loads per wave and step
    constexpr int STG = ROWS * BK;                        // halfs per stage
    constexpr int NQ = BK / 16;                           // 16-wide pieces of a step
    static_assert(ROWS % (RPI * NW) == 0 && BN % RPI == 0, "whole load instructions");
    static_assert(EPI != kGemmSwiglu && EPI != kGemmQKV ? true : TN % 2 == 0, "pairs of groups");
    __shared__ __attribute__((aligned(1024))) f16 ring[NS * STG];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WN, wm = wave / WN;
    const int h = lane >> 5, col = lane & 31;

    // Workgroup i runs on XCD i % 8: each XCD takes a contiguous range of tiles,
    // prompt rows fastest, so that its L2 holds its own weights ...
    const int T = a.n_tiles * a.m_tiles;
    const int per = (T + 7) / 8;
    const int tile = static_cast<int>(blockIdx.x & 7) * per + static_cast<int>(blockIdx.x >> 3);
    if (static_cast<int>(blockIdx.x >> 3) >= per || tile >= T) return;
    // ... in bands of at most 8 row tiles: the 32 tiles an XCD works on at once
    // then share 4 tiles of weights and 8 of rows instead of 2 and 16, and a weight
    // is read by one XCD a band.
    const int gm = min(a.m_tiles, 8);
    const int band = tile / (gm * a.n_tiles), in_band = tile % (gm * a.n_tiles);
    const int bm = min(gm, a.m_tiles - band * gm);
    const int n0 = in_band / bm * BN, m0 = (band * gm + in_band % bm) * BM;

    // weight row of local row r
    auto wrow = [&](int r) {
        const int gl = (n0 + r) / 32, i = r % 32;
        if constexpr (EPI == kGemmSwiglu) {
            const int half = a.N / 2;
            return min(gl / 2 * 32 + i, half - 1) + (gl & 1) * half;
        } else if constexpr (EPI == kGemmQKV) {
            const int ppd = a.D / 64;
            return min(gl / 2 / ppd * a.D + gl / 2 % ppd * 32 + i + (gl & 1) * (a.D / 2), a.N - 1);
        } else {
            return min(n0 + r, a.N - 1);
        }
    };
    const int k0 = static_cast<int>(blockIdx.y) * a.k_steps;   // this K range's first step
    // chunk c of row r sits at c ^ swz(r): 16 neighbouring rows of one chunk
    // cover a 256-byte bank line's 16 slots
    auto swz = [](int r) { return CPR == 8 ? r >> 1 & 7 : r >> 2 & 3; };
    const int KT = min(a.k_steps, a.K / BK - k0);
    const uint32_t ring0 = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((lds_void*)(lds_f16*)ring));

    // per-lane source offsets of this wave's loads (bytes)
    uint32_t voff[LPT];
#pragma unroll
    for (int p = 0; p < LPT; ++p) {
        const int r = (wave * LPT + p) * RPI + lane / CPR;
        const int c = lane % CPR ^ swz(r);
        const int row = r < BN ? wrow(r) : min(m0 + r - BN, a.M - 1);
        voff[p] = static_cast<uint32_t>(row) * static_cast<uint32_t>(2 * a.K) + 16 * c;
    }
    auto issue = [&](int slot, int t, int p) {   // load p of step t
        const int inst = wave * LPT + p;         // uniform
        const f16* base = (inst * RPI < BN ? a.W : a.A) + (k0 + t) * BK;
        dma16s(base, voff[p], ring0 + (slot * STG + inst * RPI * BK) * 2);
    };
    // operand reads: rows of this wave's tiles at chunk 2q + h of piece q
    const int wr0 = (wn * TN * 32 + col) * BK, mr0 = (BN + wm * TM * 32 + col) * BK;
    static_assert(BN % 32 == 0 && BM % 32 == 0, "whole 32-row groups");
    int sw[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) sw[q] = 8 * ((2 * q + h) ^ swz(col));
    half8 w2[2][TN], m2[2][TM];
    // operand r of piece q: the first MFMA's two first
    auto read = [&](const f16* s, int q, int r, half8 (&w)[TN], half8 (&m)[TM]) {
        if (r == 0 || r > TM)
            w[r ? r - TM : 0] = *reinterpret_cast<const half8*>(s + wr0 + 32 * (r ? r - TM : 0) * BK + sw[q]);
        else
            m[r - 1] = *reinterpret_cast<const half8*>(s + mr0 + 32 * (r - 1) * BK + sw[q]);
    };
    floatx16 acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    // The MFMAs of one piece.  The next piece's operand reads and this piece's
    // share of the loads go out behind its first MFMAs, one or two at a time:
    // issued as a block they held both waves of a SIMD off the matrix cores.
    constexpr int MF = TN * TM, R = TN + TM;
    constexpr int RPM = (R + (MF > 2 ? MF - 2 : 1) - 1) / (MF > 2 ? MF - 2 : 1);
    auto mma = [&](const half8 (&w)[TN], const half8 (&m)[TM], auto&& after) {
#pragma unroll
        for (int x = 0; x < MF; ++x) {
            acc[x / TM][x % TM] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[x / TM], m[x % TM], acc[x / TM][x % TM], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            after(x);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // The residual of this lane's outputs, read ahead of the ring's loads (after
    // the products it cost 5 us of an o projection at 2048 rows): 8 columns
    // 8(u + h) .. +8 of row col, as store8 writes them.
    const int mw = m0 + wm * TM * 32 + col;
    u32x4 resid[EPI == kGemmResidual ? TN * TM * 2 : 1];
    if constexpr (EPI == kGemmResidual) {
#pragma unroll
        for (int x = 0; x < TN * TM * 2; ++x) {
            const int nb = min(n0 + (wn * TN + x / 2 / TM) * 32, a.N - 32), u = 2 * (x % 2);
            const int m = min(mw + 32 * (x / 2 % TM), a.M - 1);
            resid[x] = *reinterpret_cast<const u32x4*>(a.out + (int64_t)m * a.N + nb + 8 * (u + h));
        }
    }

#pragma unroll
    for (int t = 0; t < NS - 1; ++t)
        if (t < KT)
#pragma unroll
            for (int p = 0; p < LPT; ++p) issue(t, t, p);
    if (KT >= NS - 1)
        wait_vm<(NS - 2) * LPT>();
    else
        wait_vm<0>();
    stage_barrier();
    int slot = 0;                        // of step t
#pragma unroll
    for (int r = 0; r < R; ++r) read(ring, 0, r, w2[0], m2[0]);
    constexpr int LQ = (LPT + NQ - 2) / (NQ - 1);   // loads per piece but the last
    auto step = [&](int t, bool ld, bool more) {
        const int prev = slot == 0 ? NS - 1 : slot - 1;
        const f16* st = ring + slot * STG;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const f16* from = st;
            if (q + 1 == NQ && more) {
                // this wave's loads of step t+1 (exact while later steps follow)
                if (ld)
                    wait_vm<(NS - 2) * LPT>();
                else
                    wait_vm<0>();
                stage_barrier();
                slot = slot + 1 == NS ? 0 : slot + 1;
                from = ring + slot * STG;
            }
            const int nq = (q + 1) % NQ;
            const int p0 = q * LQ, np = q + 1 < NQ ? min(LQ, LPT - p0) : 0;
            mma(w2[q & 1], m2[q & 1], [&](int x) {
                if (q + 1 < NQ || more)
#pragma unroll
                    for (int r = x * RPM; r < (x + 1) * RPM && r < R; ++r)
                        read(from, nq, r, w2[nq & 1], m2[nq & 1]);
                if (ld)
#pragma unroll
                    for (int p = 0; p < LQ; ++p)
                        if (p < np && p * MF / LQ == x) issue(prev, t + NS - 1, p0 + p);
            });
        }
    };
    static_assert(NQ % 2 == 0, "operand buffers alternate");
    int t = 0;
    for (; t + NS - 1 < KT; ++t) step(t, true, true);
    for (; t + 1 < KT; ++t) step(t, false, true);
    step(t, false, false);

    // ---- epilogue: lane (h, col) holds W rows 8u + 4h .. +4 (u = 0..3) of each
    //      group for prompt row col of each row tile.  Two u's swap halves across
    //      the wave, so that a lane stores 8 consecutive columns, 8(u + h) ..+8.
    auto store8 = [&](f16* p, half4 x, half4 y) {   // p: columns 8(u + h)
        const uint2 xa = __builtin_bit_cast(uint2, x), ya = __builtin_bit_cast(uint2, y);
        auto s0 = __builtin_amdgcn_permlane32_swap(xa.x, ya.x, false, false);
        auto s1 = __builtin_amdgcn_permlane32_swap(xa.y, ya.y, false, false);
        *reinterpret_cast<u32x4*>(p) = u32x4{s0[0], s1[0], s0[1], s1[1]};
    };
    if constexpr (EPI == kGemmSwiglu || EPI == kGemmQKV) {
#pragma unroll
        for (int i = 0; i < TN; i += 2) {
            const int pr = (n0 + wn * TN * 32) / 64 + i / 2;   // pair of groups
            if constexpr (EPI == kGemmSwiglu) {
                if (pr * 64 >= a.N) continue;
#pragma unroll
                for (int j = 0; j < TM; ++j) {
                    const int m = mw + 32 * j;
#pragma unroll
                    for (int u = 0; u < 4; u += 2) {
                        half4 o[2];
#pragma unroll
                        for (int v = 0; v < 2; ++v)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                o[v][e] = static_cast<f16>(silu_mul(
                                    r16(acc[i][j][4 * (u + v) + e]), r16(acc[i + 1][j][4 * (u + v) + e])));
                        if (m < a.M)
                            store8(a.out + (int64_t)m * (a.N / 2) + pr * 32 + 8 * (u + h), o[0], o[1]);
                    }
                }
            } else {
                const int half = a.D / 2, ppd = a.D / 64;
                const int head = pr / ppd;
                if (head >= a.Hq + 2 * a.Hkv) continue;
                const bool isq = head < a.Hq, rot = head < a.Hq + a.Hkv;
                const int hh = isq ? head : rot ? head - a.Hq : head - a.Hq - a.Hkv;
                f16* base = (isq ? a.out : rot ? a.k : a.v) + hh * a.D;
                const int pitch = (isq ? a.Hq : a.Hkv) * a.D;
                const int d0 = pr % ppd * 32;
#pragma unroll
                for (int j = 0; j < TM; ++j) {
                    const int m = mw + 32 * j;
                    floatx4 cs[4][2];   // the row's rotations, all in flight at once
                    const floatx4* rp = reinterpret_cast<const floatx4*>(
                        a.rope + (int64_t)min(m, a.M - 1) * half + d0 + 4 * h);
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        cs[u][0] = rp[4 * u];
                        cs[u][1] = rp[4 * u + 1];
                    }
#pragma unroll
                    for (int u = 0; u < 4; u += 2) {
                        half4 o1[2], o2[2];
#pragma unroll
                        for (int v = 0; v < 2; ++v) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float x1 = r16(acc[i][j][4 * (u + v) + e]);
                                const float x2 = r16(acc[i + 1][j][4 * (u + v) + e]);
                                const float c = cs[u + v][e / 2][2 * (e & 1)], s = cs[u + v][e / 2][2 * (e & 1) + 1];
                                o1[v][e] = static_cast<f16>(rot ? x1 * c - x2 * s : x1);
                                o2[v][e] = static_cast<f16>(rot ? x2 * c + x1 * s : x2);
                            }
                        }
                        if (m < a.M) {
                            f16* p = base + (int64_t)m * pitch + d0 + 8 * (u + h);
                            store8(p, o1[0], o1[1]);
                            store8(p + half, o2[0], o2[1]);
                        }
                    }
                }
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const int nb = n0 + (wn * TN + i) * 32;   // N % 32 == 0: whole groups
            if (nb >= a.N) continue;
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                const int m = mw + 32 * j;
                if constexpr (EPI == kGemmF32) {
                    float* p = a.out32 + ((int64_t)blockIdx.y * a.M + m) * a.N + nb + 4 * h;
                    if (m < a.M)
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            *reinterpret_cast<floatx4*>(p + 8 * u) =
                                floatx4{acc[i][j][4 * u], acc[i][j][4 * u + 1], acc[i][j][4 * u + 2],
                                        acc[i][j][4 * u + 3]};
                    continue;
                }
                f16* p = a.out + (int64_t)m * a.N + nb;
#pragma unroll
                for (int u = 0; u < 4; u += 2) {
                    // back to this lane's columns: 8u + 4h .. +4 and 8(u + 1) + 4h .. +4
                    const u32x4 rr = resid[(i * TM + j) * 2 + u / 2];
                    auto s0 = __builtin_amdgcn_permlane32_swap(rr[0], rr[2], false, false);
                    auto s1 = __builtin_amdgcn_permlane32_swap(rr[1], rr[3], false, false);
                    const half4 r[2] = {__builtin_bit_cast(half4, uint2{s0[0], s1[0]}),
                                        __builtin_bit_cast(half4, uint2{s0[1], s1[1]})};
                    half4 o[2];
#pragma unroll
                    for (int v = 0; v < 2; ++v)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o[v][e] = static_cast<f16>(acc[i][j][4 * (u + v) + e] + static_cast<float>(r[v][e]));
                    if (m < a.M) store8(p + 8 * (u + h), o[0], o[1]);
                }
            }
        }
    }
}

// out[i] = fp16(sum over K ranges in order + out[i]), 8 columns a thread.
constexpr int kMaxRanges = 8;
__global__ void __launch_bounds__(256)
gemm_reduce_kernel(const float* part, f16* out, uint32_t chunks, int ranges) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= chunks) return;
    floatx4 p[kMaxRanges][2];
#pragma unroll
    for (int r = 0; r < kMaxRanges; ++r)
        if (r < ranges) {
            const floatx4* src = reinterpret_cast<const floatx4*>(part + ((int64_t)r * chunks + t) * 8);
            p[r][0] = src[0];
            p[r][1] = src[1];
        }
    half8 o = load_half8(out + 8 * (int64_t)t);
    floatx4 v0 = p[0][0], v1 = p[0][1];
#pragma unroll
    for (int r = 1; r < kMaxRanges; ++r)
        if (r < ranges) {
            v0 += p[r][0];
            v1 += p[r][1];
        }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        o[e] = static_cast<f16>(v0[e] + static_cast<float>(o[e]));
        o[4 + e] = static_cast<f16>(v1[e] + static_cast<float>(o[4 + e]));
    }
    store_half8(out + 8 * (int64_t)t, o);
}

// The tile for a shape: the smallest estimate over four tiles of rounds x
// (start and end of a workgroup + steps x time of a step).  The step times (us)
// were measured on weights that no cache holds, as a model meets them (one set
// after another, 700 MB in all): few workgroups resident, and every slot taken,
// where the L2 -> CU path is shared; between the two they are interpolated, but
// for the 64 x 64 tile, which shares a CU (and its path) from the 257th
// workgroup on.  On warm weights the same steps take .50-.75, .28-.46, .19-.27 and
// .21-.28, and a choice by those ran 320-700 rows on 128 x 64 tiles, slower than
// rocBLAS.  Us in the table's order, then rocBLAS without the epilogue's work:
//   rows   down 2048 x 5632           o 2048 x 2048              QKV 2560 x 2048
//    320   74 / 45 / 40 / 29 | 29     28 / 18 / 16 / 13 | 13     31 / 20 / 17 / 14 | 13
//    512   79 / 53 / 40 / 30 | 29     30 / 20 / 16 / 13 | 13     33 / 22 / 17 / 18 | 15
//   1024   77 / 52 / 40 / 43 | 40     30 / 21 / 16 / 17 | 17     33 / 23 / 32 / 30 | 23
//   2048   75 / 57 / 78 / 85 | 58     30 / 24 / 31 / 33 | 25     33 / 43 / 47 / 47 | 29
// gate/up 11264 x 2048: 33 rows 29 / 20 / 19 / 16 | 16, 256 33 / 24 / 33 / 36 | 28,
// 512 34 / 43 / 47 / 51 | 32, 2048 102 / 126 / 163 / 174 | 88.
struct GemmTile {
    int bn, bm, slots;
    float lo, hi;
};
constexpr GemmTile kTiles[] = {
    {256, 128, 256, 0.80f, 1.00f},
    {128, 128, 256, 0.46f, 0.62f},
    {128, 64, 256, 0.40f, 0.42f},
    {64, 64, 512, 0.30f, 0.45f},
};
constexpr float kTileEnds = 3.f;   // us: first loads, epilogue
constexpr int kNumCUs = 256;

int gemm_pick(int M, int N, int K) {
    int best = 0;
    float cost = 0.f;
    for (int i = 0; i < 4; ++i) {
        const GemmTile& c = kTiles[i];
        const int64_t T = (int64_t)((N + c.bn - 1) / c.bn) * ((M + c.bm - 1) / c.bm);
        const int64_t rounds = (T + c.slots - 1) / c.slots;
        const float full = std::min(1.f, static_cast<float>(T) / static_cast<float>(c.slots));
        const float share = c.slots > kNumCUs ? (T > kNumCUs ? 1.f : 0.f)
                                              : std::max(0.f, (full - 0.25f) / 0.75f);
        const float step = c.lo + (c.hi - c.lo) * share;
        const float t = static_cast<float>(rounds) * (kTileEnds + step * static_cast<float>(K / 64));
        if (i == 0 || t < cost) {
            cost = t;
            best = i;
        }
    }
    return best;
}

template <int BN, int BM, int WN, int WM, int NS, int EPI>
void launch_tile(GemmArgs a, hipStream_t s) {
    a.n_tiles = (a.N + BN - 1) / BN;
    a.m_tiles = (a.M + BM - 1) / BM;
    const int T = a.n_tiles * a.m_tiles, steps = a.K / 64;
    if (a.k_steps == 0) a.k_steps = steps;
    hipLaunchKernelGGL((gemm_kernel<BN, BM, 64, WN, WM, NS, EPI>),
                       dim3((T + 7) / 8 * 8, (steps + a.k_steps - 1) / a.k_steps),
                       dim3(WN * WM * kWave), 0, s, a);
}

template <int EPI>
int launch_gemm(const GemmArgs& a, hipStream_t s, const char* what, int tile = -1) {
    switch (tile < 0 ? gemm_pick(a.M, a.N, a.K) : tile) {
        case 0: launch_tile<256, 128, 4, 2, 3, EPI>(a, s); break;
        case 1: launch_tile<128, 128, 2, 4, 4, EPI>(a, s); break;
        case 2: launch_tile<128, 64, 2, 2, 4, EPI>(a, s); break;
        default: launch_tile<64, 64, 1, 2, 4, EPI>(a, s); break;
    }
    return check_launch(what);
}

GemmArgs gemm_args(const void* A, const void* W, int M, int N, int K) {
    GemmArgs a{};
    a.A = static_cast<const f16*>(A);
    a.W = static_cast<const f16*>(W);
    a.M = M;
    a.N = N;
    a.K = K;
    return a;
}

}  // namespace

bool gemm_fits(int64_t M, int64_t N, int64_t K) {
    // whole steps, whole 32-row groups, 32-bit byte offsets into A and W, and a
    // tile count (64 x 64 tiles) that the grid takes
    return M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 32 == 0 && M * K < (1ll << 31) &&
           N * K < (1ll << 31) && (M + 63) / 64 * ((N + 63) / 64) < (1ll << 24);
}

// K ranges of the residual product: few 64 x 64 tiles over a long K leave most CUs
// idle, so K is cut into ranges of 8 steps or more (the last takes what is left)
// whose fp32 partial products a second launch adds in order.  Ranges x tiles is at most 256, so the partials
// fit kGemmWorkspace.
int gemm_ranges(int M, int N, int K) {
    const int T = (N + 63) / 64 * ((M + 63) / 64), steps = K / 64;
    if (T > 128 || steps < 16) return 1;
    const int want = std::min({kMaxRanges, 256 / T, steps / 8});
    const int per = (steps + want - 1) / want;
    return (steps + per - 1) / per;
}

size_t gemm_residual_workspace(int M, int N, int K) {
    const int r = gemm_ranges(M, N, K);
    return r > 1 ? sizeof(float) * (size_t)r * M * N : 0;
}

int gemm_residual(const void* A, const void* W, void* out, int M, int N, int K, void* ws,
                  size_t ws_bytes, hipStream_t s) {
    GemmArgs a = gemm_args(A, W, M, N, K);
    a.out = static_cast<f16*>(out);
    const int ranges = gemm_ranges(M, N, K);
    if (ranges == 1 || ws_bytes < gemm_residual_workspace(M, N, K))
        return launch_gemm<kGemmResidual>(a, s, "gemm_residual");
    a.out32 = static_cast<float*>(ws);
    a.k_steps = (K / 64 + ranges - 1) / ranges;
    KVHP_REQUIRE(launch_gemm<kGemmF32>(a, s, "gemm_residual", 3) == KVHP_OK, KVHP_ERR_HIP,
                 "gemm_residual: partial products");
    const uint32_t chunks = static_cast<uint32_t>((int64_t)M * N / 8);
    hipLaunchKernelGGL(gemm_reduce_kernel, dim3((chunks + 255) / 256), dim3(256), 0, s, a.out32,
                       a.out, chunks, ranges);
    return check_launch("gemm_residual (sum)");
}

int gemm_f32(const void* A, const void* W, float* out, int M, int N, int K, hipStream_t s) {
    GemmArgs a = gemm_args(A, W, M, N, K);
    a.out32 = out;
    return launch_gemm<kGemmF32>(a, s, "gemm_f32");
}

int gemm_swiglu(const void* A, const void* W_gate_up, void* out, int M, int F, int K,
                hipStream_t s) {
    GemmArgs a = gemm_args(A, W_gate_up, M, 2 * F, K);
    a.out = static_cast<f16*>(out);
    return launch_gemm<kGemmSwiglu>(a, s, "gemm_swiglu");
}

int gemm_qkv(const void* A, const void* W_qkv, const float2* rope, void* q, void* k, void* v,
             int M, int num_q_heads, int num_kv_heads, int head_dim, int K, hipStream_t s) {
    GemmArgs a = gemm_args(A, W_qkv, M, (num_q_heads + 2 * num_kv_heads) * head_dim, K);
    a.out = static_cast<f16*>(q);
    a.k = static_cast<f16*>(k);
    a.v = static_cast<f16*>(v);
    a.rope = rope;
    a.Hq = num_q_heads;
    a.Hkv = num_kv_heads;
    a.D = head_dim;
    return launch_gemm<kGemmQKV>(a, s, "gemm_qkv");
}

}  // namespace kvhp
