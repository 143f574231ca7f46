// prefill.hip -- causal flash attention for prefill on CDNA4 fp16 MFMA (gfx950).
//
// Work decomposition: a 512-thread workgroup (8 waves) owns one KV head and
// a query block of 32*RB rows for all G query heads of that KV head: G*RB
// units of (head, 32 rows).  With KG = 1 each wave owns one unit (RB = 8/G);
// with KG = 2 (G <= 4; chosen where doubling the workgroup count fills the
// CUs without adding a round, e.g. S <= 2048 at B = 1) two wave groups share
// the units and split every tile's keys.  Each 64-key K/V
// tile is read from HBM once per workgroup and consumed by all 8 waves, so
// GQA heads share their K/V traffic.  Query blocks i and N-1-i are processed
// by the same workgroup (two passes), giving every workgroup the same causal
// work (KG = 2: odd KV heads run the long block first), when those
// pairs fill the GPU; below that (S < 2048 at 32/8 heads) every block gets
// its own workgroup, longest first, so that more CUs share the work (S=512
// 15.4 vs 21.5 us).  Grid x enumerates (pair or block, kv_head) with the kv
// head fastest.
//
// K/V staging: a 4-stage LDS ring (4 x 32 KB for D=128), filled by
// global_load_lds_dwordx4 (direct HBM->LDS, no VGPR round trip).  Tile t+2 is
// issued when tile t's phases begin; before reading a stage each wave waits
// for its own loads of that stage (explicit s_waitcnt vmcnt(N)) and the
// workgroup meets at one barrier per ping-pong phase.  Rows are stored with an XOR
// swizzle of their 16-byte chunks so that both the K reads (ds_read_b128)
// and the transposing V reads (ds_read_b64_tr_b16) are bank-conflict free.
//
// Per tile and unit, on v_mfma_f32_32x32x16_f16, transposed so that one lane
// owns one query row for the whole online softmax:
//   S^T = K Q^T     A = K rows from LDS, B = Q^T held in registers.
//   softmax         fp32 in the log2 domain; the causal mask is applied only on
//                   tiles that cross the diagonal; the running max moves (and
//                   O is rescaled) only when a row's max passes it by 8 in
//                   log2 units, so P <= 256 stays exact in fp16; row sums by
//                   v_dot2_f32_f16 over the fp16 P.
//   O^T += V^T P^T  A = V^T read with ds_read_b64_tr_b16 (transposing 8-byte
//                   LDS reads), B = P^T converted to fp16 straight from the
//                   S^T accumulators.
// The tile loop is a ping-pong: waves 0-3 and 4-7 (one of each per SIMD)
// alternate an MFMA step (S^T of tile j, O^T of tile j-1, operand reads
// scheduled ahead, at wave priority 1) and a softmax step one phase apart.
//
// With 5..8 query heads per KV head the same split runs with a KV head's query
// heads on two workgroups.  A prompt's last positions behind a cached prefix
// run on the same kernel with the keys read from their pages.
//
// With a page pool, each workgroup also writes the K/V rows of its own query
// block into the pages after its outputs (every key row is written exactly
// once, bit-exact).
//
// Roofline: MFMA-bound for long prompts; algorithmic work 4*D*Hq*S(S+1)/2
// flops (the two causal contractions).
#include "kvhp_internal.h"

#include <algorithm>
#include <cmath>

namespace kvhp {

namespace {

constexpr int kBN = 64;     // keys per tile
constexpr int kNumCUs = 256;  // MI355X compute units (work-split heuristic only)

struct PrefillArgs {
    const f16* q;           // [B][S][Hq][D]
    const f16* k;           // [B][S][Hkv][D]
    const f16* v;
    f16* out;               // [B][S][Hq][D]
    f16* pool_k;            // optional page pool [Hkv][P][16][D]
    f16* pool_v;
    const int32_t* bt;      // [B][max_pages]
    int max_pages;
    int num_pages;
    int S, Hq, Hkv, G;
    int RB;                 // 16-row blocks per query block (fast kernel)
    int n_qblk;
    int paired;             // 1: query blocks i and n-1-i share a workgroup (two passes)
    float scale_log2;
    int HG, nsub;           // SUB: query heads per workgroup, workgroups per KV head
    int fold;               // unpaired, > 0: this many blocks longest first, then the others
                            // shortest first (two workgroups per CU)
    int side;               // fold: the blocks of one rank of all sequences side by side
    // CACHED: the q rows sit at positions first .. first + S - 1 and all keys are
    // read from the pages (k, v: the pools; bt, max_pages, num_pages as above).
    int first;
    int tiles_per_split;    // key tiles of a split (blockIdx.z)
    int nsplit;
    float* ws_o;            // [S * Hq][nsplit][D], nsplit > 1
    float* ws_ml;           // [S * Hq][nsplit][2]  (max in log2 units, sum)
};

typedef short short4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v lds_short4v;
typedef __attribute__((address_space(3))) f16 lds_f16;
typedef __attribute__((address_space(3))) void lds_void;

// ds_read_b64_tr_b16: within each 16-lane block, lane i receives element
// (i % 4) of the 8-byte groups addressed by lanes 4k + i/4, k = 0..3.
__device__ __forceinline__ short4v lds_read_tr16(const f16* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4v*)(lds_f16*)p);
}

__device__ __forceinline__ half8 cat_half8(short4v lo, short4v hi) {
    return __builtin_bit_cast(half8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// global_load_lds_dwordx4: lane l's 16 bytes land at lds_base + 16*l (M0
// holds the wave-uniform LDS base).  Issued as inline asm so that only the
// explicit vmcnt waits of the ring order it against the LDS reads: the
// compiler's own tracking cannot tell ring stages apart and would otherwise
// drain every in-flight stage before each read.
__device__ __forceinline__ void dma16(const f16* src, f16* lds_base) {
    const uint32_t m0v = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((lds_void*)(lds_f16*)lds_base));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :: "s"(m0v), "v"(src) : "memory", "m0");
}

// Same with a wave-uniform base in SGPRs and a 32-bit per-lane byte offset.
__device__ __forceinline__ void dma16s(const f16* sbase, uint32_t voff, f16* lds_base) {
    const uint32_t m0v = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((lds_void*)(lds_f16*)lds_base));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(m0v), "v"(voff), "s"(sbase) : "memory", "m0");
}

// s_waitcnt vmcnt(N) (expcnt / lgkmcnt left free).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// Orders this wave's LDS accesses across the barrier without the vmcnt(0)
// drain a __syncthreads() fence implies (which would empty the DMA ring).
__device__ __forceinline__ void ring_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr float kLazyLog2 = 8.f;  // P stays below 2^8 between rescales

// Sum / max across the two 32-lane halves of a wave (v_permlane32_swap).
__device__ __forceinline__ float halves_max(float x) {
    auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
    auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(t[0]) + __uint_as_float(t[1]);
}

// A workgroup of 8 waves serves one KV head and a query block of 32*RB rows
// for all G query heads of that KV head: G*RB units of (head, 32 rows).  With
// KG = 1 each wave owns one unit (G*RB <= 8); with KG = 2 (G <= 4) the waves
// form two groups of four that share the units and split every 64-key tile
// (group y takes keys 32y..32y+31), and the two softmax states of a unit are
// merged through LDS at the end -- half the query rows per workgroup, so
// twice the workgroups.  K/V tiles of 64 keys stream through a 4-stage LDS ring
// filled by direct global->LDS loads and are read by every wave, so GQA
// heads share their K/V traffic; rows are stored XOR-swizzled (16-byte
// chunk c of row r at position c ^ swz(r)) so the operand reads hit distinct
// banks without padding.  Query blocks i and N-1-i run in the same workgroup
// so every workgroup does the same causal work.
//
// Contractions on v_mfma_f32_32x32x16_f16 (lane l: row/column l%32, k-slots
// 8(l/32)..+8; accumulator element i is row 8(i/4) + 4(l/32) + i%4):
//   S^T = K Q^T     A = K rows (ds_read_b128), B = Q^T in registers; lane l
//                   owns query row l%32 of its unit, 32 of the 64 keys.
//   O^T += V^T P^T  per 16-key step t: A = V^T by two transposing 8-byte
//                   reads, B = P^T = fp16 of accumulator elements 8u..8u+7
//                   of key block t/2 (u = t%2): k-slot (h, e) is key
//                   16t + 4h + e for e < 4 and 16t + 8 + 4h + e - 4 above.
// Per 64-key tile a wave does 32 MFMAs (1 MFLOP) for 32 KB of LDS reads,
// twice the work per LDS byte of 16x16 tiles.
//
// SUB: a KV head's query heads are cut into nsub groups of at most HG, a
// workgroup each (G = 5..8 at KG = 2).
//
// CACHED: attention of a prompt's last S positions over keys in pages, the
// cached prefix included.  A tile's four pages are loaded through their ids,
// which sit in LDS from the start (a load from the block table inside the loop
// would wait for every DMA in flight).  Few query rows leave CUs idle, so the
// keys may be cut into nsplit ranges; a row whose keys reach past the first
// stores its partial (m, l, O) for prefill_merge_kernel.
// P is 0 at the keys past a row, but 0 times an infinite or NaN V is NaN, and a
// later position's V must not reach an earlier row (whose K/V stay in pages that
// other prompts share).  In the tiles that the causal mask can cut, such elements
// are set to 0 in LDS, by the wave that loaded them, and added as they are at the
// end to the rows at or past their key.  (The whole-prompt kernel does not: there
// a non-finite V also reaches the earlier rows of its block.)
constexpr int kMaxTablePages = 4088;   // page ids of a split in LDS (65408 keys) ...
constexpr int kBadWords = 8;           // ... and the keys of 4 tiles with such a V

template <int D, int KG, bool SUB, bool CACHED>
__global__ void __launch_bounds__(8 * kWave)
prefill_mfma_kernel(const PrefillArgs a) {
    constexpr int WAVES = 8;
    constexpr int UPG = WAVES / KG;     // units per wave group
    constexpr int NTH = WAVES * kWave;  // threads per workgroup
    constexpr int NC = D / 16;          // k-chunks of the QK contraction
    constexpr int NDB = D / 32;         // 32-dim blocks of the output
    constexpr int CPR = D / 8;          // 16-byte chunks per row
    constexpr int RPI = kWave / CPR;    // rows per DMA instruction
    constexpr int IPW = kBN / RPI / WAVES;  // DMA instructions per wave per matrix
    constexpr int LPT = 2 * IPW;        // DMA loads per wave per tile (K + V)
    constexpr int TB = kBN * D;         // halfs per tile matrix
    // K swizzle: 16 consecutive rows of one chunk cover the 16 slots of a
    // 256-byte bank line (D = 64: two rows a line; c ^ (r & 7) there read rows r
    // and r + 8 from the same banks, half of the LDS cycles).
    auto kswz = [](int r) { return CPR == 16 ? r & 15 : r >> 1 & 7; };
    // V swizzle: the transposing reads of one half-wave touch 4 consecutive
    // rows x 4 chunks; these land on distinct 16-byte bank groups of the
    // 256-byte bank line.
    auto vswz = [](int r) { return CPR == 16 ? 4 * (r & 3) : (r & 3) << 1; };

    constexpr int NSTAGE = 4;
    __shared__ __attribute__((aligned(16))) f16 ring[NSTAGE * 2 * TB];
    __shared__ int32_t ptab[CACHED ? kMaxTablePages + kBadWords : 1];
    uint32_t* bad_keys = reinterpret_cast<uint32_t*>(ptab + kMaxTablePages);   // CACHED

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: LDS bases in SGPRs
    const int lane = tid & 63;
    const int h = lane >> 5;        // k-slot half
    const int c32 = lane & 31;      // row / column in the 32x32 operands
    const int j16 = lane & 15;      // lane within its 16-lane block
    const int blk2 = (lane >> 4) & 1;

    const int hw = SUB ? a.Hkv * a.nsub : a.Hkv;   // workgroups per block or pair
    const int kvh = SUB ? blockIdx.x % hw / a.nsub : blockIdx.x % a.Hkv;
    const int sub = SUB ? blockIdx.x % hw % a.nsub : 0;
    // pair index (paired) or block rank, longest first, and sequence; side by side:
    // grid (KV head, group and sequence, 1, block)
    const bool side = D == 64 && KG == 2 && !CACHED && a.side;
    const int xq = blockIdx.x / hw;
    const int pair = side ? blockIdx.z : xq;
    const int b = side ? xq : blockIdx.y;
    const int S = a.S;
    const int G = SUB ? min(a.HG, a.G - sub * a.HG) : a.G;   // this workgroup's query heads
    const int head0 = kvh * a.G + sub * a.HG;                // and the first of them
    const int first = CACHED ? a.first : 0;
    const int n_keys = first + S;
    const int t_lo = CACHED ? static_cast<int>(blockIdx.z) * a.tiles_per_split : 0;
    const int RB = a.RB;
    const int BM = 32 * RB;
    const int nunits = G * RB;
    const int64_t qrs = (int64_t)a.Hq * D;     // q/out row stride
    const int64_t kvrs = (int64_t)a.Hkv * D;   // k/v row stride
    const f16* kb = CACHED ? a.k + (int64_t)kvh * a.num_pages * kPage * D
                           : a.k + (int64_t)b * S * kvrs + (int64_t)kvh * D;
    const f16* vb = CACHED ? a.v + (int64_t)kvh * a.num_pages * kPage * D
                           : a.v + (int64_t)b * S * kvrs + (int64_t)kvh * D;

    // DMA of tile tt into a stage: this wave's rows (wave*IPW + p)*RPI + lane/CPR.
    // Tiles past the last one re-load the last tile (an L2 hit): every path
    // issues the same loads, so the vmcnt bookkeeping stays exact.
    // Per-lane DMA source offsets inside a tile (bytes): row and swizzled chunk.
    uint32_t dko[IPW], dvo[IPW];
#pragma unroll
    for (int p = 0; p < IPW; ++p) {
        const int row = (wave * IPW + p) * RPI + lane / CPR;
        const int ck = (lane % CPR) ^ kswz(row);
        const int cv = (lane % CPR) ^ vswz(row);
        dko[p] = static_cast<uint32_t>((row * kvrs + 8 * ck) * 2);
        dvo[p] = static_cast<uint32_t>((row * kvrs + 8 * cv) * 2);
    }
    int last_tile = 0;
    // CACHED: this wave's 8 rows of a tile lie in page wave / 2 of its four.
    const int last_pi = (n_keys - 1) >> 4, last_slot = (n_keys - 1) & 15;
    int pid_next = 0;   // page id of the next issue, read one issue ahead
    auto page_of = [&](int tt) { return min((t_lo + min(tt, last_tile)) * 4 + (wave >> 1), last_pi); };
    auto issue = [&](f16* stg, int tt) {
        if constexpr (CACHED) {
            // rows past the context's last token re-read its row (finite)
            const int pu = (t_lo + min(tt, last_tile)) * 4 + (wave >> 1);
            const int lim = pu >= last_pi ? last_slot : kPage - 1;
            const int64_t page = (int64_t)__builtin_amdgcn_readfirstlane(pid_next) * (kPage * D);
#pragma unroll
            for (int p = 0; p < IPW; ++p) {
                const int blk = wave * IPW + p;
                const int row = blk * RPI + lane / CPR;
                const uint32_t src = static_cast<uint32_t>(min(row & (kPage - 1), lim) * D * 2);
                dma16s(kb + page, src + 16 * ((lane % CPR) ^ kswz(row)), stg + blk * RPI * D);
                dma16s(vb + page, src + 16 * ((lane % CPR) ^ vswz(row)), stg + TB + blk * RPI * D);
            }
            pid_next = ptab[page_of(tt + 1) - t_lo * 4];
            return;
        }
        tt = min(tt, last_tile);
        const int key0 = tt * kBN;
        if (key0 + kBN <= S) {
            const f16* kt = kb + (int64_t)key0 * kvrs;
            const f16* vt = vb + (int64_t)key0 * kvrs;
#pragma unroll
            for (int p = 0; p < IPW; ++p) {
                const int blk = wave * IPW + p;
                dma16s(kt, dko[p], stg + blk * RPI * D);
                dma16s(vt, dvo[p], stg + TB + blk * RPI * D);
            }
        } else {
            // the last, partial tile: rows past the prompt re-read row S-1
#pragma unroll
            for (int p = 0; p < IPW; ++p) {
                const int blk = wave * IPW + p;
                const int row = blk * RPI + lane / CPR;
                const int key = min(key0 + row, S - 1);
                const int ck = (lane % CPR) ^ kswz(row);
                const int cv = (lane % CPR) ^ vswz(row);
                dma16(kb + (int64_t)key * kvrs + 8 * ck, stg + blk * RPI * D);
                dma16(vb + (int64_t)key * kvrs + 8 * cv, stg + TB + blk * RPI * D);
            }
        }
    };
    // Per-lane LDS read offsets (halfs) inside a stage: K operand chunk c of
    // key row 32*kgrp + c32 (+32 per extra key block), and V^T operand of dim
    // block db at key row 32*kgrp + 4h + j16/4 (+16 per key step, +8 for the
    // second read).  The swizzles depend on the lane only.
    const int kgrp_ = wave / (WAVES / KG);
    int kro[NC], vro[NDB];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int r = 32 * kgrp_ + c32;
        kro[c] = r * D + 8 * ((2 * c + h) ^ kswz(r));
    }
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
        const int R1 = 32 * kgrp_ + 4 * h + j16 / 4;
        const int ch = 4 * db + 2 * blk2 + ((j16 & 3) >> 1);
        vro[db] = R1 * D + 8 * (ch ^ vswz(R1)) + 4 * (j16 & 1);
    }

    for (int pass = 0; pass < 2; ++pass) {
        // KG = 2: odd KV heads (other XCDs) take their long block
        // first, so that half the workgroups load Q and drain stores while
        // the other half run tile loops (every workgroup of a KV head still
        // walks the same tiles together).
        const bool flip = KG == 2 && (kvh & 1) != 0;
        int qblk;
        if (a.paired) {
            qblk = (pass == 0) != flip ? pair : a.n_qblk - 1 - pair;
            if (pass == 1 && a.n_qblk - 1 - pair <= pair) break;   // odd count: middle block once
        } else {
            if (pass == 1) break;
            qblk = a.n_qblk - 1 - pair;   // one block per workgroup, longest first
            if (D == 64 && KG == 2)
                if (a.fold && pair >= a.fold) qblk = pair - a.fold;
        }
        const int q0 = qblk * BM;

        // ---- this wave's unit: head kvh*G + u%G, rows r0 .. r0+31; its key
        //      half of every tile (all 64 keys when KG == 1)
        const int u = wave % UPG;
        const int kgrp = wave / UPG;
        const bool uvalid = u < nunits;
        const int qh = (SUB ? head0 : kvh * G) + (uvalid ? u % G : 0);
        const int r0 = q0 + 32 * (uvalid ? u / G : 0);
        const int row = r0 + c32;
        half8 qop[NC];
        {
            const bool live = uvalid && row < S;
            const f16* qp = a.q + ((int64_t)b * S + row) * qrs + (int64_t)qh * D + 8 * h;
#pragma unroll
            for (int c = 0; c < NC; ++c) qop[c] = live ? load_half8(qp + 16 * c) : half8{};
        }
        floatx16 o[NDB];
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
        float m_run = -1e30f, l_part = 0.f;
        const float lazy_thr = kLazyLog2 / a.scale_log2;   // in raw score units

        const int last_row = min(q0 + BM, S) - 1;
        int n_tiles = (first + last_row) / kBN + 1;
        if constexpr (CACHED) {
            n_tiles = min(n_tiles - t_lo, a.tiles_per_split);
            if (n_tiles <= 0) return;   // the block's keys end before this split
        }
        last_tile = n_tiles - 1;
        if constexpr (CACHED) {
            // the split's page ids, clamped into the pool
            const int np = min(n_tiles * 4, last_pi - t_lo * 4 + 1);
            for (int i = tid; i < np; i += NTH) {
                const int pid = t_lo * 4 + i < a.max_pages ? a.bt[t_lo * 4 + i] : 0;
                ptab[i] = min(max(pid, 0), a.num_pages - 1);
            }
            if (tid < kBadWords) bad_keys[tid] = 0;
            __syncthreads();
            pid_next = ptab[page_of(0) - t_lo * 4];
        }

        wait_vmcnt<0>();  // q in registers before the ring: no compiler waits inside it
        ring_barrier();   // everyone is done with the previous pass's stages
        issue(ring, 0);
        issue(ring + 2 * TB, 1);

        constexpr int NKB = 2 / KG;     // this wave's 32-key blocks per tile
        auto qk = [&](const f16* Kt, floatx16 (&sc)[NKB]) {
#pragma unroll
            for (int kb2 = 0; kb2 < NKB; ++kb2) {
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[kb2][i] = 0.f;
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const half8 kop = *reinterpret_cast<const half8*>(&Kt[kro[c] + 32 * kb2 * D]);
                    sc[kb2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kop, qop[c], sc[kb2], 0, 0, 0);
                }
            }
        };
        floatx16 sc[NKB];
        half8 pop[2 * NKB];
#pragma unroll
        for (int kb2 = 0; kb2 < NKB; ++kb2)
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[kb2][i] = 0.f;
#pragma unroll
        for (int t = 0; t < 2 * NKB; ++t) pop[t] = half8{};

        // Ping-pong: the two wave groups (waves 0-3, 4-7; one wave of each per
        // SIMD; with KG = 2 the two key halves of every tile) alternate an
        // MFMA step and a softmax step, group 1 one phase behind group 0, so
        // that one wave's MFMAs run under the other's exponentials.  The
        // barriers order memory only, so the compiler may still move a step's
        // ALU work across them; the MFMA step's operand reads are scheduled PF
        // ahead of their MFMAs.  With the MFMA step at wave priority 1 this
        // beats a plain per-tile loop (QK of tile t+1, softmax of t, PV of t in
        // every wave) at every size: S=2048 45.4 vs 47.1 us, S=8192 516 vs
        // 540 us.
        //   mstep(j): S^T(j) = K(j) Q^T (j < n),  O^T += V(j-1)^T P(j-1)^T (j >= 1)
        //   sstep(j): P(j) from S^T(j); O, l rescaled when the max moves.
        // Phase 2j: group 0 mstep(j), group 1 sstep(j-1); phase 2j+1: group 0
        // sstep(j), group 1 mstep(j); one workgroup barrier between phases.
        // Ring: tile j+2 is issued at the start of phase 2j into the stage
        // of tile j-2, whose last reader (group 1's mstep(j-1)) ran in phase
        // 2j-1; before the barrier into phase 2j each wave waits for its own
        // DMA of tile j (tile j+1 may stay in flight).  Tiles past the end
        // re-load the last tile, so every wave issues the same loads.
        auto pv = [&](int j) {
            const f16* Vt = ring + (j % NSTAGE) * 2 * TB + TB;
#pragma unroll
            for (int t = 0; t < 2 * NKB; ++t) {
#pragma unroll
                for (int db = 0; db < NDB; ++db) {
                    const f16* p1 = &Vt[vro[db] + 16 * t * D];
                    const half8 vop = cat_half8(lds_read_tr16(p1), lds_read_tr16(p1 + 8 * D));
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vop, pop[t], o[db], 0, 0, 0);
                }
            }
        };
        // Operand reads run PF reads ahead of the MFMAs that use them.
        constexpr int NQK = NKB * NC, NPV = 2 * NKB * NDB;   // MFMAs
        constexpr int PF = 8;
        // The MFMA step runs at wave priority 1: when the SIMD's other wave
        // (softmax step) and this one both can issue, the MFMAs go first
        // (S=8192 516 vs 524 us, S=2048 45.4 vs 47.2 us).
        auto mstep = [&](int j) {   // 1 <= j < n_tiles
            __builtin_amdgcn_s_setprio(1);
            qk(ring + (j % NSTAGE) * 2 * TB, sc);
            pv(j - 1);
            __builtin_amdgcn_sched_group_barrier(0x100, PF, 0);
#pragma unroll
            for (int i = 0; i < NQK - PF; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
#pragma unroll
            for (int i = 0; i < NPV; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, NQK + NPV - (NQK - PF) - NPV, 0);
            __builtin_amdgcn_s_setprio(0);
        };
        auto sstep = [&](int j) {
            const int k0 = (t_lo + j) * kBN;
            const bool act = uvalid && k0 <= first + r0 + 31;
            // ---- online softmax of query row `row`; P^T operands straight
            // from S^T.  Inactive units (invalid, or entirely above the
            // diagonal) see only -inf scores: alpha = 1 and p = 0 leave their
            // state as is.  The running max is kept on raw scores and the
            // scale folded into the exponent.
            if (!act || k0 + kBN - 1 > first + r0) {
                // element (kb2, i) holds key k0 + 32(kb2 + kgrp) + 4h +
                // 8(i/4) + i%4; keys past min(row, S-1) are masked
                const int lim = act ? min(first + row, n_keys - 1) - (k0 + 32 * kgrp + 4 * h) : -1;
#pragma unroll
                for (int kb2 = 0; kb2 < NKB; ++kb2)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (32 * kb2 + 8 * (i / 4) + (i % 4) > lim) sc[kb2][i] = -INFINITY;
            }
            float tmax = -INFINITY;
#pragma unroll
            for (int kb2 = 0; kb2 < NKB; ++kb2)
#pragma unroll
                for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, sc[kb2][i]);
            tmax = halves_max(tmax);
            // Lazy rescale: m_run is a reference max, moved (and O, l
            // rescaled) only when some row's max exceeds it by more than
            // kLazyLog2 in log2 units; otherwise p = 2^(s*c - m_run*c) stays
            // below 2^kLazyLog2, exact in fp16.
            if (__builtin_amdgcn_read_exec() & __ballot(tmax > m_run + lazy_thr)) {
                const float mn = fmaxf(m_run, tmax);
                const float alpha = fast_exp2((m_run - mn) * a.scale_log2);
                l_part *= alpha;
#pragma unroll
                for (int db = 0; db < NDB; ++db) o[db] *= alpha;
                m_run = mn;
            }
            const float nmc = -m_run * a.scale_log2;
#pragma unroll
            for (int t = 0; t < 2 * NKB; ++t)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    pop[t][e] = static_cast<f16>(
                        fast_exp2(fmaf(sc[t / 2][8 * (t % 2) + e], a.scale_log2, nmc)));
            // Row sum of the fp16 P actually fed to the PV contraction, two
            // values per v_dot2_f32_f16 with fp32 accumulation.
            const half2v ones = {static_cast<f16>(1.f), static_cast<f16>(1.f)};
#pragma unroll
            for (int t = 0; t < 2 * NKB; ++t)
#pragma unroll
                for (int e = 0; e < 8; e += 2)
                    l_part = __builtin_amdgcn_fdot2(half2v{pop[t][e], pop[t][e + 1]}, ones, l_part,
                                                    false);
        };
        // CACHED: from tile cut0 on the causal mask can cut a tile (at most 3 of
        // the block's); this wave's rows of it, just landed, lose the elements of V
        // that are not finite.
        const int cut0 = (first + q0) / kBN - t_lo;
        auto clean = [&](int j) {
            f16* Vt = ring + (j % NSTAGE) * 2 * TB + TB + wave * IPW * RPI * D + 8 * lane;
            asm volatile("" ::: "memory");
#pragma unroll
            for (int p = 0; p < IPW; ++p) {
                u32x4 x = *reinterpret_cast<const u32x4*>(Vt + p * RPI * D);
                uint32_t m[4], any = 0;   // bits 15 / 31: an exponent of all ones
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    m[i] = ((x[i] & 0x7fff7fffu) + 0x04000400u) & 0x80008000u;
                    any |= m[i];
                }
                if (any == 0) continue;
                const int r = (wave * IPW + p) * RPI + lane / CPR;
                atomicOr(&bad_keys[2 * (j - cut0) + (r >> 5)], 1u << (r & 31));
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] &= ~(m[i] | (m[i] - (m[i] >> 15)));
                *reinterpret_cast<u32x4*>(Vt + p * RPI * D) = x;
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): written before the barrier
        };
        auto phase_start = [&](int j) {   // barrier into phase 2j, then tile j+2
            wait_vmcnt<LPT>();
            if (CACHED && j >= cut0 && j < n_tiles) clean(j);
            ring_barrier();
            const int tt = j + 2;
            issue(ring + (tt % NSTAGE) * 2 * TB, tt);
        };
        if ((wave >> 2) == 0) {
            phase_start(0);
            qk(ring, sc);
            ring_barrier();
            sstep(0);
            for (int j = 1; j < n_tiles; ++j) {
                phase_start(j);
                mstep(j);
                ring_barrier();
                sstep(j);
            }
            phase_start(n_tiles);
            pv(n_tiles - 1);
            ring_barrier();
        } else {
            phase_start(0);
            ring_barrier();
            qk(ring, sc);
            for (int j = 1; j < n_tiles; ++j) {
                phase_start(j);
                sstep(j - 1);
                ring_barrier();
                mstep(j);
            }
            phase_start(n_tiles);
            sstep(n_tiles - 1);
            ring_barrier();
            pv(n_tiles - 1);
        }
        wait_vmcnt<0>();  // drain the ring's trailing re-loads

        // ---- pages: this query block's own K/V rows, once per KV head.  Rows
        //      of the pass's last tile come from its ring stage (still intact:
        //      the trailing re-loads go to the other stages), earlier rows
        //      (blocks longer than a tile) from memory.
        if (!CACHED && a.pool_k && (!SUB || sub == 0)) {
            const int lt0 = last_tile * kBN;
            const f16* Ks = ring + (last_tile % NSTAGE) * 2 * TB;
            const f16* Vs = Ks + TB;
            for (int idx = tid; idx < BM * CPR; idx += NTH) {
                const int key = q0 + idx / CPR;
                const int ch = idx % CPR;
                if (key >= S || key / kPage >= a.max_pages) continue;
                const int pid = a.bt[(int64_t)b * a.max_pages + key / kPage];
                if (pid < 0 || pid >= a.num_pages) continue;
                const int64_t dst =
                    (((int64_t)kvh * a.num_pages + pid) * kPage + key % kPage) * D + 8 * ch;
                half8 kk, vv;
                if (key >= lt0) {
                    const int r = key - lt0;
                    kk = *reinterpret_cast<const half8*>(&Ks[r * D + 8 * (ch ^ kswz(r))]);
                    vv = *reinterpret_cast<const half8*>(&Vs[r * D + 8 * (ch ^ vswz(r))]);
                } else {
                    kk = load_half8(kb + (int64_t)key * kvrs + 8 * ch);
                    vv = load_half8(vb + (int64_t)key * kvrs + 8 * ch);
                }
                store_half8(a.pool_k + dst, kk);
                store_half8(a.pool_v + dst, vv);
            }
        }

        if constexpr (KG == 2) {
            // ---- group 1 hands its (m, l, O) to group 0 through the ring's
            //      LDS (every wave is past its last read of the ring).
            float* xo = reinterpret_cast<float*>(ring);
            float* xml = xo + UPG * NDB * 16 * kWave;
            ring_barrier();
            if (kgrp == 1) {
#pragma unroll
                for (int db = 0; db < NDB; ++db)
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4) {
                        floatx4 v4 = {o[db][4 * q4], o[db][4 * q4 + 1], o[db][4 * q4 + 2],
                                      o[db][4 * q4 + 3]};
                        *reinterpret_cast<floatx4*>(
                            &xo[(((u * NDB + db) * 4 + q4) * kWave + lane) * 4]) = v4;
                    }
                xml[(u * kWave + lane) * 2] = m_run;
                xml[(u * kWave + lane) * 2 + 1] = l_part;
            }
            ring_barrier();
            if (kgrp == 0) {
                const float m1 = xml[(u * kWave + lane) * 2];
                const float l1 = xml[(u * kWave + lane) * 2 + 1];
                const float mn = fmaxf(m_run, m1);
                const float a0 = fast_exp2((m_run - mn) * a.scale_log2);
                const float a1 = fast_exp2((m1 - mn) * a.scale_log2);
                if constexpr (CACHED) m_run = mn;   // O and l are relative to it from here
                l_part = l_part * a0 + l1 * a1;
#pragma unroll
                for (int db = 0; db < NDB; ++db)
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4) {
                        const floatx4 v4 = *reinterpret_cast<const floatx4*>(
                            &xo[(((u * NDB + db) * 4 + q4) * kWave + lane) * 4]);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o[db][4 * q4 + e] = o[db][4 * q4 + e] * a0 + v4[e] * a1;
                    }
            }
        }

        if constexpr (CACHED) {
            // ---- the V elements left out above, from the pages
            uint32_t any = 0;
#pragma unroll
            for (int i = 0; i < kBadWords; ++i) any |= bad_keys[i];
            if (__builtin_amdgcn_readfirstlane(any) && kgrp == 0) {
#pragma unroll 1
                for (int i = 0; i < 32 * kBadWords; ++i) {
                    const int key = (t_lo + cut0) * kBN + i;
                    if (!(bad_keys[i >> 5] >> (i & 31) & 1) || key >= n_keys) continue;
                    const f16* src = vb + ((int64_t)ptab[(key >> 4) - t_lo * 4] * kPage + key % kPage) * D + 4 * h;
#pragma unroll
                    for (int db = 0; db < NDB; ++db)
#pragma unroll
                        for (int q4 = 0; q4 < 4; ++q4) {
                            const half4 v = *reinterpret_cast<const half4*>(src + 32 * db + 8 * q4);
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float x = static_cast<float>(v[e]);
                                if (key <= first + row && !(fabsf(x) < INFINITY))
                                    o[db][4 * q4 + e] += x;
                            }
                        }
                }
            }
        }

        // ---- normalise and store: lane holds row `row`, dims 32db + 8q + 4h + e.
        {
            const float lt = halves_sum(l_part);
            // a row whose keys reach past one split leaves its partial for the merge
            const int per_split = CACHED ? a.tiles_per_split * kBN : 0;
            if (CACHED && kgrp == 0 && uvalid && row < S && first + row >= per_split) {
                // (splits past the row's keys are not read by the merge)
                const int64_t prow = ((int64_t)row * a.Hq + qh) * a.nsplit + blockIdx.z;
                float* po = a.ws_o + prow * D + 4 * h;
#pragma unroll
                for (int db = 0; db < NDB; ++db)
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4)
                        *reinterpret_cast<floatx4*>(po + 32 * db + 8 * q4) =
                            floatx4{o[db][4 * q4], o[db][4 * q4 + 1], o[db][4 * q4 + 2],
                                    o[db][4 * q4 + 3]};
                if (h == 0) {
                    a.ws_ml[prow * 2] = m_run * a.scale_log2;
                    a.ws_ml[prow * 2 + 1] = lt;
                }
            } else if (kgrp == 0 && uvalid && row < S && (!CACHED || blockIdx.z == 0)) {
                const float inv = lt > 0.f ? 1.f / lt : 0.f;
                f16* orow = a.out + ((int64_t)b * S + row) * qrs + (int64_t)qh * D + 4 * h;
#pragma unroll
                for (int db = 0; db < NDB; ++db)
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4) {
                        half4 hv;
#pragma unroll
                        for (int e = 0; e < 4; ++e) hv[e] = static_cast<f16>(o[db][4 * q4 + e] * inv);
                        *reinterpret_cast<half4*>(orow + 32 * db + 8 * q4) = hv;
                    }
            }
        }

        wait_vmcnt<0>();   // page and output stores complete before the next ring starts
    }
}

// Log-sum-exp merge of the key splits' partials, 8 dims of one (row, head) a
// thread; rows whose keys lie in the first split were written directly.  One
// workgroup per (head, row) as decode's merges take 20 us more at 512 rows of
// 32 heads.
__global__ void __launch_bounds__(256)
prefill_merge_kernel(const float* ws_o, const float* ws_ml, f16* out, int64_t threads, int Hq,
                     int D, int first, int keys_per_split, int nsplit) {
    const int64_t t = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (t >= threads) return;
    const int cpr = D / 8, c = static_cast<int>(t % cpr);
    const int64_t rh = t / cpr;
    const int n = static_cast<int>((first + rh / Hq + keys_per_split) / keys_per_split);   // its splits
    if (n <= 1) return;
    const float* po = ws_o + rh * nsplit * D + 8 * c;
    const float2* pml = reinterpret_cast<const float2*>(ws_ml) + rh * nsplit;
    float M = -3.0e38f, L = 0.f;
    floatx4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = o0;
    constexpr int U = 4;   // splits in flight
    for (int j0 = 0; j0 < n; j0 += U) {
        float2 ml[U];
        floatx4 x[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = min(j0 + u, n - 1);
            ml[u] = pml[j];
            x[u][0] = *reinterpret_cast<const floatx4*>(po + (int64_t)j * D);
            x[u][1] = *reinterpret_cast<const floatx4*>(po + (int64_t)j * D + 4);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (j0 + u >= n) continue;
            const float mn = fmaxf(M, ml[u].x);
            const float al = fast_exp2(M - mn), be = fast_exp2(ml[u].x - mn);
            o0 = o0 * al + x[u][0] * be;
            o1 = o1 * al + x[u][1] * be;
            L = fmaf(L, al, ml[u].y * be);
            M = mn;
        }
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    half8 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        h[e] = static_cast<f16>(o0[e] * inv);
        h[4 + e] = static_cast<f16>(o1[e] * inv);
    }
    store_half8(out + rh * D + 8 * c, h);
}

// Any head_dim <= 256 / any alignment: one wave per (query head, row),
// online softmax over keys 0..row.  Optionally writes the page pool too
// (from the first query head of each group, one wave per key row).
__global__ void __launch_bounds__(kWave)
prefill_generic_kernel(const PrefillArgs a, int D) {
    const int lane = threadIdx.x;
    const int qh = blockIdx.x;
    const int row = blockIdx.y;
    const int b = blockIdx.z;
    const int kvh = qh / a.G;
    const int S = a.S;
    const int64_t qrs = (int64_t)a.Hq * D, kvrs = (int64_t)a.Hkv * D;
    const f16* qp = a.q + ((int64_t)b * S + row) * qrs + (int64_t)qh * D;
    const f16* kb = a.k + (int64_t)b * S * kvrs + (int64_t)kvh * D;
    const f16* vb = a.v + (int64_t)b * S * kvrs + (int64_t)kvh * D;
    if (a.pool_k && qh % a.G == 0 && row / kPage < a.max_pages) {
        int pid = a.bt[(int64_t)b * a.max_pages + row / kPage];
        if (pid >= 0 && pid < a.num_pages) {
            const int64_t dst = (((int64_t)kvh * a.num_pages + pid) * kPage + row % kPage) * D;
            for (int d = lane; d < D; d += kWave) {
                a.pool_k[dst + d] = kb[(int64_t)row * kvrs + d];
                a.pool_v[dst + d] = vb[(int64_t)row * kvrs + d];
            }
        }
    }
    float qv[4], acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int d = lane + kWave * i;
        qv[i] = d < D ? static_cast<float>(qp[d]) : 0.f;
        acc[i] = 0.f;
    }
    float m = -1e30f, l = 0.f;
    for (int t = 0; t <= row; ++t) {
        float dot = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = lane + kWave * i;
            if (d < D) dot = fmaf(qv[i], static_cast<float>(kb[(int64_t)t * kvrs + d]), dot);
        }
        dot = wave_sum(dot);
        const float sc = dot * a.scale_log2;
        const float mn = fmaxf(m, sc);
        const float al = fast_exp2(m - mn);
        const float p = fast_exp2(sc - mn);
        l = l * al + p;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = lane + kWave * i;
            const float vv = d < D ? static_cast<float>(vb[(int64_t)t * kvrs + d]) : 0.f;
            acc[i] = fmaf(p, vv, acc[i] * al);
        }
        m = mn;
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    f16* op = a.out + ((int64_t)b * S + row) * qrs + (int64_t)qh * D;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int d = lane + kWave * i;
        if (d < D) op[d] = static_cast<f16>(acc[i] * inv);
    }
}

}  // namespace

int prefill_impl(const void* q, const void* k, const void* v, void* out, int64_t seq_len,
                 int hq, int hkv, int d, int batch, void* pool_k, void* pool_v,
                 const int32_t* bt, int max_pages, int num_pages, hipStream_t s) {
    if (seq_len <= 0 || batch <= 0) return KVHP_OK;
    KVHP_REQUIRE(q && k && v && out, KVHP_ERR_INVALID, "flash_prefill: null pointer");
    KVHP_REQUIRE(hq > 0 && hkv > 0 && hq % hkv == 0, KVHP_ERR_INVALID,
                 "flash_prefill: num_q_heads=%d must be a positive multiple of num_kv_heads=%d",
                 hq, hkv);
    KVHP_REQUIRE(d > 0 && d <= 256, KVHP_ERR_UNSUPPORTED,
                 "flash_prefill: head_dim=%d outside 1..256", d);
    KVHP_REQUIRE(seq_len <= (int64_t)1 << 30, KVHP_ERR_UNSUPPORTED,
                 "flash_prefill: seq_len %lld too large", (long long)seq_len);
    if (pool_k || pool_v || bt) {
        KVHP_REQUIRE(pool_k && pool_v && bt && max_pages > 0 && num_pages > 0,
                     KVHP_ERR_INVALID, "flash_prefill_paged: incomplete page pool arguments");
        KVHP_REQUIRE((int64_t)max_pages * kPage >= seq_len, KVHP_ERR_INVALID,
                     "flash_prefill_paged: %d pages per sequence cannot hold %lld tokens",
                     max_pages, (long long)seq_len);
    }
    PrefillArgs a{};
    a.q = static_cast<const f16*>(q);
    a.k = static_cast<const f16*>(k);
    a.v = static_cast<const f16*>(v);
    a.out = static_cast<f16*>(out);
    a.pool_k = static_cast<f16*>(pool_k);
    a.pool_v = static_cast<f16*>(pool_v);
    a.bt = bt;
    a.max_pages = max_pages;
    a.num_pages = num_pages;
    a.S = static_cast<int>(seq_len);
    a.Hq = hq;
    a.Hkv = hkv;
    a.G = hq / hkv;
    a.scale_log2 = 1.4426950408889634f / std::sqrt(static_cast<float>(d));
    a.RB = 1;
    a.n_qblk = 0;
    a.paired = 1;

    const bool fast = (d == 64 || d == 128) && a.G <= 8 && aligned16(q) && aligned16(k) &&
                      aligned16(v) && aligned16(out) &&
                      (!pool_k || (aligned16(pool_k) && aligned16(pool_v)));
    if (fast) {
        // units of (head, 32 rows) per workgroup: one per wave, or (G <= 4)
        // one per pair of waves that split each tile's keys (KG = 2: twice
        // the workgroups, each with half the rows).  A KG = 2 workgroup takes
        // ~57 % of a KG = 1 workgroup's time, so KG = 2 pays when doubling
        // the workgroups adds no round of CUs: with grid1 block pairs of one
        // unit per wave, up to half the CUs (grid1 <= 128) or one and a half
        // rounds (257..384).  Measured at 32/8 heads, D = 128: KG = 1 is
        // 12-32 % faster at grid1 = 144..256 (S = 2304..4096 at B = 1,
        // S = 1280..2048 at B = 2), 10 % at 448 and 8 % at 512; KG = 2 is
        // 19 % faster at 128 (S = 2048) and 1-10 % at 288..384.
        const int64_t qblk1 = (seq_len + 32 * (8 / a.G) - 1) / (32 * (8 / a.G));
        const int64_t grid1 = (int64_t)hkv * ((qblk1 + 1) / 2) * batch;
        const bool split = grid1 <= kNumCUs / 2 || (grid1 > kNumCUs && grid1 <= kNumCUs * 3 / 2);
        // G = 5..8 take the same split with the heads cut in two (SUB).  Us before
        // and after at D = 64: 14/2 heads 3 x 777 21.6 / 16.9, 512 15.3 / 12.0,
        // 2048 45.4 / 34.3, 4096 84.5 / 65.3; 32/4 heads 1024 24.3 / 17.5, 2048
        // 41.8 / 31.8; at D = 128, 32/4 heads 2048 59.5 / 47.5, 6000 345 / 325;
        // outside the rule (32/4 x 64 at 4096 and 8192) it is 2-4 % slower.
        const bool sub = a.G > 4 && split;
        const int kg = sub || ((a.G == 1 || a.G == 2 || a.G == 4) && split) ? 2 : 1;
        a.nsub = sub ? 2 : 1;
        a.HG = (a.G + a.nsub - 1) / a.nsub;
        a.RB = sub ? 1 : 8 / kg / a.G;
        const int bm = 32 * a.RB;
        a.n_qblk = static_cast<int>((seq_len + bm - 1) / bm);
        // pair the causal blocks only when the pairs fill every CU
        const int64_t pgrid = (int64_t)hkv * a.nsub * ((a.n_qblk + 1) / 2) * batch;
        a.paired = (pgrid >= kNumCUs) ? 1 : 0;
        // D = 64 at KG = 2 keeps two workgroups on a CU (64 KB LDS, 125 VGPRs):
        // while every block is resident at once, a block each, as many of the
        // longest as there are CUs longest first, then the others shortest first,
        // so that a CU's two add up alike (32/8 heads 2048 34.5 paired / 32.6, 32/4
        // heads 33.1 / 31.8).  A batch goes block by block, its sequences side by
        // side: one sequence after another a CU met two long blocks (32/8 heads,
        // 2 x 1000 26.7 / 21.3, paired 22.5; 3 x 333 11.6 / 10.4, paired 10.5; 4 x
        // 512 18.2 / 15.0, paired 17.0).
        const int64_t side = (int64_t)hkv * a.nsub * batch;   // workgroups per block rank
        const int blocks = a.paired ? (a.n_qblk + 1) / 2 : a.n_qblk;
        dim3 grid(hkv * a.nsub * blocks, batch);
        if (d == 64 && kg == 2 && side * a.n_qblk <= 2 * kNumCUs) {
            a.paired = 0;
            a.fold = std::max(1, static_cast<int>(kNumCUs / side));
            a.side = batch > 1;
            grid = a.side ? dim3(static_cast<unsigned>(side), 1, a.n_qblk)
                          : dim3(hkv * a.nsub * a.n_qblk);
        }
        const dim3 blk(8 * kWave);
        auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, grid, blk, 0, s, a); };
        if (d == 64)
            sub ? launch(prefill_mfma_kernel<64, 2, true, false>)
                : kg == 2 ? launch(prefill_mfma_kernel<64, 2, false, false>)
                          : launch(prefill_mfma_kernel<64, 1, false, false>);
        else
            sub ? launch(prefill_mfma_kernel<128, 2, true, false>)
                : kg == 2 ? launch(prefill_mfma_kernel<128, 2, false, false>)
                          : launch(prefill_mfma_kernel<128, 1, false, false>);
        return check_launch("flash_prefill");
    }
    dim3 grid(hq, static_cast<unsigned>(seq_len), batch);
    hipLaunchKernelGGL(prefill_generic_kernel, grid, dim3(kWave), 0, s, a, d);
    return check_launch("flash_prefill(generic)");
}

// The cached-prefix plan: query blocks of 32 rows (KG = 2), all of a block's
// keys in one split when the blocks fill the CUs, else in ranges of at least 4
// tiles so that about kNumCUs workgroups run.  Two layers with 512 new tokens
// behind 1488 cached (32/4 heads of 64) in us, aiming at 128 / 256 / 512 / 1024
// workgroups: 327 / 317 / 323 / 356 (489 as decode rows, which read the keys once
// per query row).
struct CachedPlan {
    int nsub, HG, RB, n_qblk, nsplit, tiles;
};

static bool cached_plan(int rows, int first, int hq, int hkv, int d, CachedPlan& p) {
    const int G = hq / hkv;
    if ((d != 64 && d != 128) || G > 8 || G == 3) return false;
    p.nsub = G > 4 ? 2 : 1;
    p.HG = (G + p.nsub - 1) / p.nsub;
    p.RB = G > 4 ? 1 : 4 / G;
    p.n_qblk = (rows + 32 * p.RB - 1) / (32 * p.RB);
    const int64_t wgs = (int64_t)hkv * p.nsub * p.n_qblk;
    const int tiles = (first + rows + kBN - 1) / kBN;
    int n = static_cast<int>(std::min<int64_t>(kNumCUs / std::max<int64_t>(wgs, 1), tiles / 4));
    n = std::max(n, (tiles * 4 + kMaxTablePages - 1) / kMaxTablePages);   // page ids in LDS
    n = std::max(n, 1);
    p.tiles = (tiles + n - 1) / n;
    p.nsplit = (tiles + p.tiles - 1) / p.tiles;
    return p.nsplit <= 64;
}

size_t prefill_cached_workspace(int rows, int first, int hq, int hkv, int d) {
    CachedPlan p;
    if (!cached_plan(rows, first, hq, hkv, d, p) || p.nsplit == 1) return 0;
    return sizeof(float) * (size_t)rows * hq * p.nsplit * (d + 2);
}

bool prefill_cached_fits(int rows, int first, int hq, int hkv, int d) {
    CachedPlan p;
    return cached_plan(rows, first, hq, hkv, d, p);
}

int prefill_cached(const void* q, const void* pool_k, const void* pool_v, const int32_t* bt,
                   int max_pages, int num_pages, void* out, int rows, int first,
                   int hq, int hkv, int d, void* ws, size_t ws_bytes, hipStream_t s) {
    CachedPlan p;
    KVHP_REQUIRE(cached_plan(rows, first, hq, hkv, d, p), KVHP_ERR_UNSUPPORTED,
                 "prefill_cached: %d rows behind %d keys, heads %d/%d of %d", rows, first, hq, hkv, d);
    KVHP_REQUIRE(ws_bytes >= prefill_cached_workspace(rows, first, hq, hkv, d), KVHP_ERR_WORKSPACE,
                 "prefill_cached: workspace too small");
    PrefillArgs a{};
    a.q = static_cast<const f16*>(q);
    a.k = static_cast<const f16*>(pool_k);
    a.v = static_cast<const f16*>(pool_v);
    a.out = static_cast<f16*>(out);
    a.bt = bt;
    a.max_pages = max_pages;
    a.num_pages = num_pages;
    a.S = rows;
    a.Hq = hq;
    a.Hkv = hkv;
    a.G = hq / hkv;
    a.RB = p.RB;
    a.n_qblk = p.n_qblk;
    a.scale_log2 = 1.4426950408889634f / std::sqrt(static_cast<float>(d));
    a.HG = p.HG;
    a.nsub = p.nsub;
    a.first = first;
    a.tiles_per_split = p.tiles;
    a.nsplit = p.nsplit;
    a.ws_o = static_cast<float*>(ws);
    a.ws_ml = a.ws_o + (size_t)rows * hq * p.nsplit * d;
    const dim3 grid(hkv * p.nsub * p.n_qblk, 1, p.nsplit);
    if (d == 64)
        hipLaunchKernelGGL((prefill_mfma_kernel<64, 2, true, true>), grid, dim3(8 * kWave), 0, s, a);
    else
        hipLaunchKernelGGL((prefill_mfma_kernel<128, 2, true, true>), grid, dim3(8 * kWave), 0, s, a);
    const int rc = check_launch("prefill_cached");
    if (rc || p.nsplit == 1) return rc;
    const int64_t threads = (int64_t)rows * hq * (d / 8);
    hipLaunchKernelGGL(prefill_merge_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)),
                       dim3(256), 0, s, a.ws_o, a.ws_ml, a.out, threads, hq, d, first,
                       p.tiles * kBN, p.nsplit);
    return check_launch("prefill_cached (merge)");
}

}  // namespace kvhp

using namespace kvhp;

extern "C" int kvhp_flash_prefill(const void* q, const void* k, const void* v, void* out,
                                  int64_t seq_len, int num_q_heads, int num_kv_heads,
                                  int head_dim, int batch, void* stream) {
    clear_error();
    return prefill_impl(q, k, v, out, seq_len, num_q_heads, num_kv_heads, head_dim, batch,
                        nullptr, nullptr, nullptr, 0, 0, static_cast<hipStream_t>(stream));
}

extern "C" int kvhp_flash_prefill_paged(const void* q, const void* k, const void* v,
                                        void* out, int64_t seq_len, int num_q_heads,
                                        int num_kv_heads, int head_dim, int batch,
                                        void* pool_k, void* pool_v,
                                        const int32_t* block_tables, int max_pages,
                                        int num_pages, void* stream) {
    clear_error();
    KVHP_REQUIRE(pool_k && pool_v && block_tables, KVHP_ERR_INVALID,
                 "flash_prefill_paged: null page pool / block table");
    return prefill_impl(q, k, v, out, seq_len, num_q_heads, num_kv_heads, head_dim, batch,
                        pool_k, pool_v, block_tables, max_pages, num_pages,
                        static_cast<hipStream_t>(stream));
}

extern "C" int kvhp_causal_gqa(const void* q, const void* k, const void* v, void* out,
                               int64_t seq_len, int64_t num_q_heads, int64_t num_kv_heads,
                               int64_t head_dim, void* stream) {
    clear_error();
    if (seq_len <= 0) return KVHP_OK;  // causal_attention.cu:133
    KVHP_REQUIRE(num_q_heads > 0 && num_q_heads < (1 << 20) && num_kv_heads > 0 &&
                     num_kv_heads < (1 << 20) && head_dim > 0 && head_dim < (1 << 20),
                 KVHP_ERR_INVALID, "causal_gqa: bad shape");
    return prefill_impl(q, k, v, out, seq_len, static_cast<int>(num_q_heads),
                        static_cast<int>(num_kv_heads), static_cast<int>(head_dim), 1, nullptr,
                        nullptr, nullptr, 0, 0, static_cast<hipStream_t>(stream));
}
