// D1 -- DeepSeek sparse attention (MLA absorbed) decode.
//
// The paged bf16 entry (the fp32 one: dsa_f32.hip).
// Reference: dsa_forward (kernels/dsa/naive_dsa.cu:435-474) gathers the
// selected K_c/K_p/V rows into [Q,S,*] fp32 buffers, materialises a
// [Q,H,S] score matrix, scales it, softmaxes it serially per (q,h) and
// multiplies by the gathered V; the CPU copy is tests/test_dsa.cu:23-68:
//   s = (dot(q_nope,K_c[i]) + dot(q_pe,K_p[i])) * (1/sqrt(Dc+Dp))
//   P = softmax_S(s);  out = sum_s P*V[i]
//
// The BASELINE decode (Dc=512, Dp=64, bf16 paged latent cache, V = K_c).
//   Nothing is materialised: a workgroup takes a group of heads of a query
//   over a share of its selected positions (dsa_split_kernel below),
//   translates the indices through the page table, streams 32-token tiles of
//   1152-byte latent rows into LDS, and computes per wave (16 heads)
//     S^T = K . Q^T      (bf16 MFMA; K rows from LDS, q held in registers)
//     online softmax per head (lane = head; reduction over lanes/regs)
//     O^T += V^T . P^T   (bf16 MFMA; P^T is already in the B-operand layout
//                         because S^T's output layout gives each lane the
//                         8 tokens {4g..4g+3, 16+4g..16+4g+3} of its head)
//   V^T fragments are read from the same row-major tile with the gfx950
//   transposing LDS read.  dsa_merge_kernel adds the shares up.
#include "internal.hpp"

#include <float.h>

namespace amdmoe {

// ---------------------------------------------------------------- bf16 paged
// Geometry: Dc = 512, Dp = 64, one latent row = 576 bf16 = 1152 bytes = 72
// chunks of 16 bytes.
// Out-of-range voffset for the cache loads: at least the buffer size (the
// cache is at most kMaxCacheBytes) and far enough below 2^32 that adding the
// largest soffset and the 16-byte access cannot wrap back into range.
constexpr uint32_t kOobDsa = 0xFFFFF000u;
constexpr long kMaxCacheBytes = 0xFFFFE000L;
constexpr int kDc = 512, kDp = 64, kDt = 576;
constexpr int kRowBytes = kDt * 2;               // 1152
// The most positions of one split of a group of 32, 64 or 96 heads, and so the
// most selected positions per query where H is no multiple of 128.
constexpr int kMaxS = 4096;

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Reductions over the lanes l, l^16 (resp. l^32) with the gfx950 lane
// swaps: permlane16_swap exchanges the odd 16-lane rows of its first operand
// with the even rows of its second, permlane32_swap the upper half of the
// first with the lower half of the second; with both operands the same
// value the two results hold, at every lane, the values of l and l^16
// (resp. l^32) in some order.
__device__ __forceinline__ float xor16_max(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor16_sum(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float xor32_sum(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;

// ------------------------------------------------------ split kernel
// dsa_split_kernel (H a multiple of 128): one workgroup per (query, group
// of 128 heads, token split), 8 waves; wave w owns heads 16w..16w+15 of the
// group for all of the split's tokens, so its softmax state is private (no
// exchange between waves) and P goes from the S^T accumulators straight
// into the PV MFMA operand.  32-token tiles stream through a 4-stage LDS
// ring (each tile's loads go out two tiles ahead), filled by direct
// global->LDS loads; each wave reads every tile once for S and once for V.
// dsa_split96/64/32_kernel are the same body with 6, 4 and 2 waves, for groups
// of that many heads (of any H, a multiple of 128 too, where the plan below
// finds them faster): no skew between waves, so a 3-stage ring and room for the
// rows of 4096 positions.  A wave alone on its SIMD waits for LDS and for its
// own softmax (1.5 us per tile for 0.45 of MFMAs), and with 32 heads half of
// the SIMDs have none: dsa_split32x2_kernel gives every second tile to a second
// pair of waves and adds the two sums up in LDS at the end.  One split of 32 heads
// over 2048 positions: 103.9 -> 59.5 us (Q=1), 216 -> 186 (Q=300).
//   S^T (16 tokens x 16 heads) = K . Q^T   16x16x32 bf16, 2 token tiles,
//                                          q of the wave's 16 heads in
//                                          registers
//   online softmax per head in the exp2 domain; l is kept per lane and
//     reduced once at the end
//   O^T (512 dims x 16 heads) += V^T . P^T  16x16x32 bf16 in the token
//     order of S^T's output layout: lane (head c, group g) holds tokens
//     4g..4g+3 and 16+4g..16+4g+3, and the transposed LDS reads of V^T
//     fetch the same tokens
// Registers: O is 128 accumulators and q 72, so a wave fits in 256
// registers and two waves share each SIMD (one wave's softmax, LDS waits
// and barrier run under the other's MFMAs).  The price is LDS traffic:
// every wave reads each tile for its 16 heads, 544 KB per CU per tile.  The
// running max m is raised only when a tile max exceeds it by more than 8
// (so p <= 256), and then O and l are multiplied by 2^(m_old - m_new) in
// registers; with O(1) scores the first tile's max is never exceeded by 8.
// Every split writes its unnormalised O (bf16: the output is bf16 and the
// merge sums at most a few splits in fp32) and (max, sum) per head;
// dsa_merge_kernel combines the splits and writes bf16.
//
// Tile layout (tile32_off): 1 KB blocks of 16 tokens x 4 chunks (16-byte
// chunk j of the 1152-byte row), blocks [token group][chunk group], within a
// block [token][slot] with slot = (j & 3) ^ (token bits 1-2).  Measured with
// the bank-conflict counter on gfx950, this is free of conflicts for both the
// 16-token S fragment reads (ds_read_b128, lane = token, one chunk) and the
// transposed V^T reads (ds_read_b64_tr_b16, 4 tokens x 2 chunks per 16
// lanes); XOR-ing token bits 2-3 instead (the plain 64-bank model's answer)
// cost the S reads 4 conflict cycles each.
constexpr int kT32 = 32;
constexpr int kStage32 = kT32 * kRowBytes;                // 36864
constexpr int kMaxSplitS = 65536;                         // selected positions per query (32 splits)
constexpr int kTileBlocks = kStage32 / 1024;              // 36 DMA instructions per tile
constexpr int kTrans = 4;                                 // positions per thread and round of the translation
template <int NH, int TG> struct SplitGeom {              // TG groups of NH waves
    static constexpr int RING = NH == 8 ? 4 : (TG > 1 ? 2 : 3);  // stages per group
    static constexpr int CHUNK = NH == 8 ? 2048 : (TG > 1 ? 3072 : kMaxS);  // most tokens per split
    static constexpr int ROUND = kTrans * 64 * NH * TG;   // positions the workgroup translates per round
    static constexpr int ROWS = TG * RING * kStage32;     // LDS offsets: the tokens' cache rows,
    static constexpr int MASK = ROWS + CHUNK * 4;         // their validity bits, 64 per word:
    // a round writes all of its words, past the split too (6 waves: 3 rounds
    // of 1536 positions for 4096)
    static constexpr int LDS = MASK + (CHUNK + ROUND - 1) / ROUND * (ROUND / 8);
    static_assert(LDS <= 160 * 1024 && MASK % 8 == 0, "split kernel LDS");
};

__device__ __forceinline__ int tile32_off(int t, int j) {  // token t (0..31), chunk j (0..71)
    return ((t >> 4) * 18 + (j >> 2)) * 1024 + (t & 15) * 64 + (((j & 3) ^ ((t >> 1) & 3)) << 4);
}

// 1152 zero bytes: the latent row an invalid position reads when the cache
// is addressed with 64-bit pointers (caches beyond the 4 GiB that a buffer
// descriptor's 32-bit offsets reach)
static __device__ __align__(16) uint16_t g_dsa_zero_row[kDt];

// WIDE: the cache is addressed with 64-bit per-lane pointers
// (global_load_lds_dwordx4) instead of a buffer descriptor's 32-bit offsets.
// The body is a device template behind plain kernels (the host side
// dropped the launch stub of a templated kernel instantiation using buffer
// descriptors).
//
// With nsplit == 1 the workgroup has all of the query's positions and writes
// the output rows; otherwise it writes its partial, (max, sum) per head and
// the unnormalised O: bf16 for 128-head groups (the merge adds at most a few
// in fp32), fp32 for the smaller ones.
template <bool WIDE, int NH, int TG>
__device__ __forceinline__ void dsa_split_body(
    const uint16_t* __restrict__ qn, const uint16_t* __restrict__ qp,
    const uint16_t* __restrict__ cache, long cache_bytes, const int* __restrict__ page_table,
    const int* __restrict__ logical, uint16_t* __restrict__ out, void* __restrict__ part,
    float* __restrict__ part_ml, int Q, int H, int S, int page, int pages_per_seq, int nsplit, int chunk,
    float scale_log2) {
    using G = SplitGeom<NH, TG>;
    constexpr int NW = NH * TG, kHeads = 16 * NH, kThreads = 64 * NW, kRing32 = G::RING;
    constexpr int kAhead = kRing32 > 2 ? 2 : 1;  // tiles loaded ahead
    constexpr int kBlocks = kTileBlocks / NH;    // DMA instructions per wave and tile (8 waves: 4 or 5)
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    int* s_rows = (int*)(smem + G::ROWS);
    unsigned long long* s_mask = (unsigned long long*)(smem + G::MASK);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hw = TG > 1 ? wave % NH : wave, tg = TG > 1 ? wave / NH : 0;  // heads and token group
    uint8_t* const ring = smem + tg * kRing32 * kStage32;
    // work item lin = (query, head group, split), dealt to the 8 XCDs in
    // contiguous chunks (workgroup b runs on XCD b % 8): the splits of a
    // query share an XCD, so its q rows come from HBM once and its partials
    // are written and merged within one L2
    const int hgroups = H / kHeads;
    const int per = gridDim.x / 8;
    const int lin = (blockIdx.x % 8) * per + blockIdx.x / 8;
    const int sp = lin % nsplit;
    const int qh = lin / nsplit;
    const int hg = qh % hgroups, qi = qh / hgroups;
    if (qi >= Q) return;  // padding of the grid to a multiple of 8
    const int t0 = sp * chunk;
    const int len = max(0, min(S, t0 + chunk) - t0);
    const int g = lane >> 4, c16 = lane & 15;
    const int hbase = kHeads * hg + 16 * hw;  // this wave's first head

    // Prologue, ordered so the q loads overlap the two dependent loads of
    // the page-table translation: logical indices, then page-table entries,
    // then q (18 loads per lane), then wait for all but the q loads.  The
    // q loads are waited for (by the compiler) at tile 0's first S step.
    // A token is valid when its logical index lies in [0, pages_per_seq *
    // page), its page id is >= 0 and its row inside the cache; an invalid
    // one (e.g. the -1 padding of a sequence shorter than the selection)
    // reads no page-table entry, loads a zero row and scores -inf.
    constexpr int kPer = kTrans;
    const int* lg = logical + (size_t)qi * S + t0;
    const int* pt = page_table + (size_t)qi * pages_per_seq;
    const long seq = (long)pages_per_seq * page;
    const long cache_rows = cache_bytes / kRowBytes;
    int li[kPer], pg[kPer];
    auto lookup = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int i = r0 + tid + kThreads * k;
            li[k] = i < len ? lg[i] : -1;
        }
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const bool ok = li[k] >= 0 && li[k] < seq;
            if (!ok) li[k] = -1;
            pg[k] = ok ? pt[li[k] / page] : -1;
        }
    };
    auto to_rows = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int i = r0 + tid + kThreads * k;
            const long row = (long)pg[k] * page + (li[k] >= 0 ? li[k] % page : 0);
            const bool ok = li[k] >= 0 && pg[k] >= 0 && row < cache_rows;
            if (i < len) s_rows[i] = ok ? (int)row : -1;
            // validity of split tokens r0 + 64(NW k + w) .. +63 (none past len)
            const unsigned long long m = __ballot(ok);
            if (lane == 0) s_mask[r0 / 64 + NW * k + wave] = m;
        }
    };
    // (8 waves take a split's 2048 positions in one round)
    if constexpr (NH < 8)
        for (int r0 = G::ROUND; r0 < len; r0 += G::ROUND) lookup(r0), to_rows(r0);
    lookup(0);
    __builtin_amdgcn_sched_barrier(0);
    // q of head hbase + c16 as B fragments: K-step ks = 32 dims, group g holds 8
    u32x4 qf[18];
    {
        const size_t hrow = (size_t)qi * H + hbase + c16;
        const uint16_t* qnr = qn + hrow * kDc;
        const uint16_t* qpr = qp + hrow * kDp;
#pragma unroll
        for (int ks = 0; ks < 16; ks++) qf[ks] = *(const u32x4*)(qnr + 32 * ks + 8 * g);
#pragma unroll
        for (int ks = 0; ks < 2; ks++) qf[16 + ks] = *(const u32x4*)(qpr + 32 * ks + 8 * g);
    }
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<18>();  // every page-table entry has arrived
    to_rows(0);
    lds_barrier();  // s_rows, s_mask visible (the q loads stay in flight)

    const __amdgpu_buffer_rsrc_t rc = make_rsrc(cache, cache_bytes);
    // DMA: block b of a tile is filled by one instruction, lane l taking
    // token 16 (b / 18) + (l >> 2), chunk 4 (b % 18) + ((l & 3) ^ ((l >> 3) & 3));
    // the chunk-group offset goes in soffset (an instruction immediate would
    // also move the LDS address)
    const uint32_t lane_c16 = 16u * (uint32_t)((lane & 3) ^ ((lane >> 3) & 3));
    using RowAddr = std::conditional_t<WIDE, const uint8_t*, uint32_t>;
    auto row_vo = [&](int tok) __attribute__((always_inline)) -> RowAddr {
        if constexpr (WIDE) {
            const uint8_t* a = (const uint8_t*)g_dsa_zero_row + lane_c16;
            if (tok < len) {
                const long r = s_rows[tok];
                const long off = r * kRowBytes + lane_c16;
                if (r >= 0 && off < cache_bytes) a = (const uint8_t*)cache + off;
            }
            return a;
        } else {
            uint32_t vo = kOobDsa;
            if (tok < len) {
                const long r = s_rows[tok];
                const long off = r * kRowBytes + lane_c16;
                if (r >= 0 && off < cache_bytes) vo = (uint32_t)off;
            }
            return vo;
        }
    };
    // a tile's 36 blocks: wave w of its group issues b = w + NH n (8 waves: n < 5
    // for waves 0-3 and n < 4 for waves 4-7)
    auto issue_blk = [&](int st, RowAddr vo0, RowAddr vo1, int n) __attribute__((always_inline)) {
        const int b = hw + NH * n;
        const int tg = b >= 18 ? 1 : 0;
        if constexpr (WIDE)
            __builtin_amdgcn_global_load_lds((gptr_t)((tg ? vo1 : vo0) + 64 * (b - 18 * tg)),
                                             (lds_ptr_t)(ring + st * kStage32 + b * 1024), 16, 0, 0);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rc, (lds_ptr_t)(ring + st * kStage32 + b * 1024), 16, tg ? vo1 : vo0, 64 * (b - 18 * tg), 0, 0);
    };
    const bool extra = kTileBlocks % NH != 0 && hw < kTileBlocks % NH;  // uniform: a fifth block per tile
    auto issue_tile = [&](int st, RowAddr vo0, RowAddr vo1) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < kBlocks; n++) issue_blk(st, vo0, vo1, n);
        if (extra) issue_blk(st, vo0, vo1, kBlocks);
    };

    f32x4 o[32];  // dims 16mt + 4g + i, head hbase + c16
#pragma unroll
    for (int i = 0; i < 32; i++) o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_lane = 0.0f;
    const int ntiles = (len + kT32 - 1) / kT32;

    const int koff = tile32_off(c16, g);  // S fragment (token tile tt, K-step ks): + 1024 (18 tt + ks)
    int vlo[2];                           // V^T read, dim tile mt: vlo[mt & 1] + 1024 (mt >> 1)
#pragma unroll
    for (int e = 0; e < 2; e++)
        vlo[e] = tile32_off(4 * g + (c16 >> 2), 2 * e + ((c16 >> 1) & 1)) + 8 * (c16 & 1);

    // The two waves of a SIMD (w and w + 4) run half a tile apart: waves
    // 0-3 pass the tile barrier at the start of a tile, waves 4-7 between
    // their S^T and PV phases, so one wave's S^T fragment reads, softmax and
    // barrier wait run under the other's PV MFMAs.  Barrier n is where waves
    // 0-3 start tile n and waves 4-7 finish S^T of tile n-1, so tile n's
    // stage is read between barriers n and n+2; the DMA of tile n+2 goes out
    // after barrier n into the stage of tile n-2 (read until barrier n), and
    // every wave waits for its blocks of tile n before barrier n.  Each wave
    // passes ntiles + 1 barriers.
    // The smaller groups have no lag: tile n is read between barriers n and
    // n+1, and tile n+2 goes into the stage of n-1.  Two token groups have a
    // ring of 2 stages each, for every second tile: tile n is their tile n/2, and
    // the next one goes into the stage of the one before.
    const bool lag = NH == 8 && wave >= 4;  // uniform
    // prologue: the first tiles (tiles past the end read zeros into their stage)
#pragma unroll
    for (int i = 0; i < kAhead; i++) {
        const int tok = kT32 * (TG * i + tg) + (lane >> 2);
        issue_tile(i, row_vo(tok), row_vo(tok + 16));
    }
    // this wave's blocks of the older of its two tiles in flight have landed
    auto wait_older = [&]() __attribute__((always_inline)) {
        if (extra) wait_vmcnt<kBlocks + 1>();
        else wait_vmcnt<kBlocks>();
    };

    // S^T (2 token tiles x 16 heads) of the tile in stage soff, 18 K-steps,
    // fragment reads kPre steps ahead; with ISSUE, one block of tile tn goes
    // out per step for the first steps
    auto s_phase = [&](auto issuec, uint32_t soff, int stn, RowAddr nvo0, RowAddr nvo1,
                       f32x4 (&sacc)[2]) __attribute__((always_inline)) {
        constexpr bool ISSUE = decltype(issuec)::value;
        const uint8_t* kb = ring + soff;
        constexpr int kPre = NW > 4 ? 2 : 6;  // (at most 4 waves: one per SIMD, with its registers)
        u32x4 a[18][2];
#pragma unroll
        for (int ks = 0; ks < kPre; ks++)
#pragma unroll
            for (int tt = 0; tt < 2; tt++) a[ks][tt] = *(const u32x4*)(kb + koff + 1024 * (18 * tt + ks));
        static_for<18>([&](auto ksc) __attribute__((always_inline)) {
            constexpr int ks = decltype(ksc)::value;
            if constexpr (ks + kPre < 18)
#pragma unroll
                for (int tt = 0; tt < 2; tt++)
                    a[ks + kPre][tt] = *(const u32x4*)(kb + koff + 1024 * (18 * tt + ks + kPre));
#pragma unroll
            for (int tt = 0; tt < 2; tt++)
                sacc[tt] = mfma_bf16(a[ks][tt], qf[ks], ks == 0 ? (f32x4){0.f, 0.f, 0.f, 0.f} : sacc[tt]);
            if constexpr (ISSUE && ks < kBlocks) issue_blk(stn, nvo0, nvo1, ks);
            if constexpr (ISSUE && ks == kBlocks)
                if (extra) issue_blk(stn, nvo0, nvo1, kBlocks);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // online softmax of tile t's scores; returns P^T as the PV B operand.
    // Lane: head c16, tokens 16tt + 4g + i of the tile; an invalid token (or
    // one past the split) scores -inf
    auto softmax = [&](int t, const f32x4 (&sacc)[2]) __attribute__((always_inline)) -> u32x4 {
        float sv[2][4], tm = -INFINITY;
        const uint32_t vmask = (uint32_t)(s_mask[t >> 1] >> (32 * (t & 1) + 4 * g));
#pragma unroll
        for (int tt = 0; tt < 2; tt++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                sv[tt][i] = (vmask >> (16 * tt + i)) & 1u ? sacc[tt][i] * scale_log2 : -INFINITY;
                tm = fmaxf(tm, sv[tt][i]);
            }
        tm = xor32_max(xor16_max(tm));
        // uniform: no valid token so far (validity is per token, the same
        // for every head)
        if (m_run == -INFINITY) {
            m_run = tm;
        } else if (__ballot(tm > m_run + 8.0f)) {
            // rare: rescale O and l to a new running max
            const float m_new = fmaxf(m_run, tm);
            const float corr = exp2f(m_run - m_new);
            l_lane *= corr;
            m_run = m_new;
#pragma unroll
            for (int mt = 0; mt < 32; mt++) o[mt] *= corr;
        }
        float p[2][4];
        // with no valid token yet every score is -inf: subtract 0, not -inf
        const float m_use = m_run == -INFINITY ? 0.0f : m_run;
#pragma unroll
        for (int tt = 0; tt < 2; tt++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                p[tt][i] = __builtin_amdgcn_exp2f(sv[tt][i] - m_use);  // 0 for a masked -inf score
                l_lane += p[tt][i];
            }
        return (u32x4){pack_bf16x2(p[0][0], p[0][1]), pack_bf16x2(p[0][2], p[0][3]),
                       pack_bf16x2(p[1][0], p[1][1]), pack_bf16x2(p[1][2], p[1][3])};
    };
    // O^T += V^T . P^T over the tile in stage soff; with ISSUE, one block of
    // tile tn goes out after each of the first 5 dim tiles
    auto pv_phase = [&](auto issuec, uint32_t soff, int stn, RowAddr nvo0, RowAddr nvo1,
                        const u32x4& pb) __attribute__((always_inline)) {
        constexpr bool ISSUE = decltype(issuec)::value;
        const uint8_t* kb = ring + soff;
        auto vfrag = [&](int mt) __attribute__((always_inline)) {
            const uint8_t* p = kb + vlo[mt & 1] + 1024 * (mt >> 1);
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)p);
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p + 18 * 1024));
            const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
            return (u32x4){l2[0], l2[1], h2[0], h2[1]};
        };
        constexpr int kPreV = NW > 4 ? 6 : 12;
        u32x4 va[32];
#pragma unroll
        for (int mt = 0; mt < kPreV; mt++) va[mt] = vfrag(mt);
        static_for<32>([&](auto mtc) __attribute__((always_inline)) {
            constexpr int mt = decltype(mtc)::value;
            if constexpr (mt + kPreV < 32) va[mt + kPreV] = vfrag(mt + kPreV);
            o[mt] = mfma_bf16(va[mt], pb, o[mt]);
            if constexpr (ISSUE && mt < kBlocks) issue_blk(stn, nvo0, nvo1, mt);
            if constexpr (ISSUE && mt == kBlocks)
                if (extra) issue_blk(stn, nvo0, nvo1, kBlocks);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto stage_of = [](int t) __attribute__((always_inline)) -> uint32_t {
        uint32_t soff = (uint32_t)(t % kRing32) * kStage32;
        asm volatile("" : "+s"(soff));
        return soff;
    };
    using on = std::integral_constant<bool, true>;
    using off = std::integral_constant<bool, false>;

    if (!lag) {
        // the q loads (older than the tile DMA) have landed: without this the
        // compiler waits for every load in flight, tile 1's included
        wait_older();
        for (int u = 0; u * TG < ntiles; u++) {  // uniform
            const int t = TG * u + tg, un = u + kAhead;
            const int tok = kT32 * (TG * un + tg) + (lane >> 2);
            const RowAddr nvo0 = row_vo(tok), nvo1 = row_vo(tok + 16);
            if constexpr (kAhead == 2) wait_older();  // tile t landed (this wave's part); tile t+1 may stay in flight
            else wait_vmcnt<0>();
            bare_barrier();  // barrier u
            if (TG == 1 || t < ntiles) {  // uniform in the wave
                const uint32_t soff = stage_of(u);
                f32x4 sacc[2];
                s_phase(on{}, soff, un % kRing32, nvo0, nvo1, sacc);
                const u32x4 pb = softmax(t, sacc);
                pv_phase(off{}, soff, 0, nvo0, nvo1, pb);
            }
        }
        if constexpr (NH == 8) bare_barrier();  // barrier ntiles
    } else {
        wait_older();
        bare_barrier();  // barrier 0
        issue_tile(2, row_vo(kT32 * 2 + (lane >> 2)), row_vo(kT32 * 2 + 16 + (lane >> 2)));
        for (int t = 0; t < ntiles; t++) {
            const int tn = t + 3;
            const RowAddr nvo0 = row_vo(kT32 * tn + (lane >> 2)), nvo1 = row_vo(kT32 * tn + 16 + (lane >> 2));
            const uint32_t soff = stage_of(t);
            f32x4 sacc[2];
            s_phase(off{}, soff, 0, nvo0, nvo1, sacc);
            const u32x4 pb = softmax(t, sacc);
            wait_older();    // tile t+1 landed (this wave's part); tile t+2 may stay in flight
            bare_barrier();  // barrier t+1
            pv_phase(on{}, soff, tn % kRing32, nvo0, nvo1, pb);
        }
    }
    wait_vmcnt<0>();  // the trailing (out-of-range) tile loads

    float l = xor32_sum(xor16_sum(l_lane));
    if constexpr (TG == 2) {  // the groups' sums, weighted as in the merge kernels
        lds_barrier();        // every wave is past its last tile
        float* xo = (float*)smem + hw * (64 * 130) + lane;  // 128 sums, max and sum per lane, 64 lanes apart
        if (tg == 1) {
#pragma unroll
            for (int i = 0; i < 128; i++) xo[64 * i] = o[i >> 2][i & 3];
            xo[64 * 128] = m_run;
            xo[64 * 129] = l;
        }
        lds_barrier();
        if (tg == 1) return;
        const float m1 = xo[64 * 128], l1 = xo[64 * 129];
        const float m = fmaxf(m_run, m1), mu = m == -INFINITY ? 0.0f : m;  // no valid position: weights 0
        const float w0 = exp2f(m_run - mu), w1 = exp2f(m1 - mu);
#pragma unroll
        for (int i = 0; i < 128; i++) o[i >> 2][i & 3] = o[i >> 2][i & 3] * w0 + xo[64 * i] * w1;
        l = l * w0 + l1 * w1;
        m_run = m;
    }
    if (NH < 8 && nsplit == 1) {  // all of the query's positions: the output rows
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        uint16_t* orow = out + ((size_t)qi * H + hbase + c16) * kDc + 4 * g;
#pragma unroll
        for (int mt = 0; mt < 32; mt++)
            *(u32x2*)(orow + 16 * mt) = (u32x2){pack_bf16x2(o[mt][0] * inv, o[mt][1] * inv),
                                                pack_bf16x2(o[mt][2] * inv, o[mt][3] * inv)};
        return;
    }
    // the split's partial in the accumulator order (each store contiguous
    // over the wave) and (max, sum) per head
    const size_t prow0 = ((size_t)qi * nsplit + sp) * H + hbase;
    if constexpr (NH == 8) {
        uint16_t* pb_base = (uint16_t*)part + prow0 * kDc + (size_t)lane * 4;
#pragma unroll
        for (int mt = 0; mt < 32; mt++)
            *(u32x2*)(pb_base + 256 * mt) =
                (u32x2){pack_bf16x2(o[mt][0], o[mt][1]), pack_bf16x2(o[mt][2], o[mt][3])};
    } else {
        float* pf = (float*)part + prow0 * kDc + (size_t)lane * 4;
#pragma unroll
        for (int mt = 0; mt < 32; mt++) *(f32x4*)(pf + 256 * mt) = o[mt];
    }
    if (g == 0) *(float2*)(part_ml + 2 * (prow0 + c16)) = make_float2(m_run, l);
}

#define AMDMOE_DSA_SPLIT_KERNEL(NAME, W, NH, TG)                                                      \
    __global__ __launch_bounds__(64 * NH * TG, 1) void NAME(                                          \
        const uint16_t* __restrict__ qn, const uint16_t* __restrict__ qp,                             \
        const uint16_t* __restrict__ cache, long cache_bytes, const int* __restrict__ page_table,     \
        const int* __restrict__ logical, uint16_t* __restrict__ out, void* __restrict__ part,         \
        float* __restrict__ part_ml, int Q, int H, int S, int page, int pages_per_seq, int nsplit,    \
        int chunk, float scale_log2) {                                                                \
        dsa_split_body<W, NH, TG>(qn, qp, cache, cache_bytes, page_table, logical, out, part,         \
                                  part_ml, Q, H, S, page, pages_per_seq, nsplit, chunk, scale_log2);  \
    }
AMDMOE_DSA_SPLIT_KERNEL(dsa_split_kernel, false, 8, 1)
AMDMOE_DSA_SPLIT_KERNEL(dsa_split_wide_kernel, true, 8, 1)
AMDMOE_DSA_SPLIT_KERNEL(dsa_split96_kernel, false, 6, 1)
AMDMOE_DSA_SPLIT_KERNEL(dsa_split64_kernel, false, 4, 1)
AMDMOE_DSA_SPLIT_KERNEL(dsa_split32_kernel, false, 2, 1)
AMDMOE_DSA_SPLIT_KERNEL(dsa_split32x2_kernel, false, 2, 2)
AMDMOE_DSA_SPLIT_KERNEL(dsa_split64_wide_kernel, true, 4, 1)
AMDMOE_DSA_SPLIT_KERNEL(dsa_split32_wide_kernel, true, 2, 1)
AMDMOE_DSA_SPLIT_KERNEL(dsa_split32x2_wide_kernel, true, 2, 2)
#undef AMDMOE_DSA_SPLIT_KERNEL

// Combines the splits of dsa_split_kernel: per (query, head), m = max of
// the split maxima, weights c_j = 2^(m_j - m), out = (sum c_j O_j) /
// (sum c_j l_j), bf16.  Workgroup = one query x 16 heads (one partial block),
// wave w = dim tiles 8w..8w+7 in the block's accumulator order: every load
// is 512 bytes contiguous, and lane (g, c) holds dims 16mt + 4g + i of head c.
// Splits are read four at a time, every load of the four in flight at once
// (one round trip for up to four splits); a later group whose maximum is
// higher rescales the sums so far by 2^(m_old - m_new).
__global__ __launch_bounds__(256) void dsa_merge_kernel(const uint16_t* __restrict__ part_b,
                                                        const float* __restrict__ part_ml,
                                                        uint16_t* __restrict__ out, int Q,
                                                        int H, int nsplit) {
    // same XCD dealing as dsa_split_kernel: a query's blocks on the XCD
    // whose L2 holds its partials
    const int h16 = H / 16;
    const int per = gridDim.x / 8;
    const int lin = (blockIdx.x % 8) * per + blockIdx.x / 8;
    const int qi = lin / h16, hb = lin % h16;
    if (qi >= Q) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, c16 = lane & 15;
    const int h = 16 * hb + c16;
    constexpr int kGroup = 4;
    f32x4 acc[8];
#pragma unroll
    for (int k = 0; k < 8; k++) acc[k] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, L = 0.0f;
    for (int j0 = 0; j0 < nsplit; j0 += kGroup) {
        float2 ml[kGroup];
        u32x2 pv[kGroup][8];
#pragma unroll
        for (int u = 0; u < kGroup; u++) {
            const int j = min(j0 + u, nsplit - 1);  // in bounds; splits past the end get weight 0
            const size_t blk = ((size_t)qi * nsplit + j) * H + 16 * hb;  // first row of the block
            ml[u] = *(const float2*)(part_ml + 2 * (blk + c16));
            const u32x2* po = (const u32x2*)(part_b + blk * kDc) + 64 * 8 * wave + lane;
#pragma unroll
            for (int k = 0; k < 8; k++) pv[u][k] = po[64 * k];
        }
        float mg = m;
#pragma unroll
        for (int u = 0; u < kGroup; u++)
            if (j0 + u < nsplit) mg = fmaxf(mg, ml[u].x);
        if (mg == -INFINITY) continue;  // no valid position so far: the sums stay 0
        // the sums so far are 0 while m = -inf
        const float r = m == -INFINITY ? 0.0f : exp2f(m - mg);
        L *= r;
#pragma unroll
        for (int k = 0; k < 8; k++) acc[k] *= r;
        m = mg;
#pragma unroll
        for (int u = 0; u < kGroup; u++) {
            const float c = j0 + u < nsplit && ml[u].x != -INFINITY ? exp2f(ml[u].x - m) : 0.0f;
            L += c * ml[u].y;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                acc[k][0] += c * __uint_as_float(pv[u][k][0] << 16);
                acc[k][1] += c * __uint_as_float(pv[u][k][0] & 0xffff0000u);
                acc[k][2] += c * __uint_as_float(pv[u][k][1] << 16);
                acc[k][3] += c * __uint_as_float(pv[u][k][1] & 0xffff0000u);
            }
        }
    }
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    uint16_t* orow = out + ((size_t)qi * H + h) * kDc + 4 * g;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int mt = 8 * wave + k;
        const u32x2 pk = {pack_bf16x2(acc[k][0] * inv, acc[k][1] * inv),
                          pack_bf16x2(acc[k][2] * inv, acc[k][3] * inv)};
        *(u32x2*)(orow + 16 * mt) = pk;
    }
}

// The same for the fp32 partials of the small head groups' kernels.  These calls are
// small (fewer than 256 head groups) and have up to a few dozen
// splits, so a workgroup is one wave per (query, 16 heads, two dim tiles),
// eight splits' loads in flight.
__global__ __launch_bounds__(64) void dsa_merge_f32_kernel(const float* __restrict__ part,
                                                           const float* __restrict__ part_ml,
                                                           uint16_t* __restrict__ out, int H, int nsplit) {
    const int mt = 2 * (blockIdx.x & 15), qh = blockIdx.x >> 4;
    const int h16 = H / 16;
    const int qi = qh / h16, hb = qh - qi * h16;
    const int lane = threadIdx.x, g = lane >> 4, c16 = lane & 15;
    constexpr int kGroup = 8;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    float m = -INFINITY, L = 0.0f;
#pragma unroll 1
    for (int j0 = 0; j0 < nsplit; j0 += kGroup) {
        float2 ml[kGroup];
        f32x4 pv[kGroup][2];
#pragma unroll
        for (int u = 0; u < kGroup; u++) {
            const int j = min(j0 + u, nsplit - 1);  // in bounds; splits past the end get weight 0
            const size_t blk = ((size_t)qi * nsplit + j) * H + 16 * hb;
            ml[u] = *(const float2*)(part_ml + 2 * (blk + c16));
            const f32x4* po = (const f32x4*)(part + blk * kDc) + 64 * mt + lane;
            pv[u][0] = po[0];
            pv[u][1] = po[64];
        }
        __builtin_amdgcn_sched_barrier(0);  // every load before the first use
        float mg = m;
#pragma unroll
        for (int u = 0; u < kGroup; u++) {
            if (j0 + u >= nsplit) ml[u].x = -INFINITY;
            mg = fmaxf(mg, ml[u].x);
        }
        const float mu = mg == -INFINITY ? 0.0f : mg;  // no valid position so far: weights 0
        const float r = exp2f(m - mu);                 // 0 while m = -inf
        m = mg;
        L *= r;
        acc[0] *= r;
        acc[1] *= r;
#pragma unroll
        for (int u = 0; u < kGroup; u++) {
            const float c = exp2f(ml[u].x - mu);
            if (j0 + u < nsplit) {  // uniform
                L += c * ml[u].y;
                acc[0] += c * pv[u][0];
                acc[1] += c * pv[u][1];
            }
        }
    }
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    uint16_t* orow = out + ((size_t)qi * H + 16 * hb + c16) * kDc + 16 * mt + 4 * g;
#pragma unroll
    for (int k = 0; k < 2; k++)
        *(u32x2*)(orow + 16 * k) = (u32x2){pack_bf16x2(acc[k][0] * inv, acc[k][1] * inv),
                                           pack_bf16x2(acc[k][2] * inv, acc[k][3] * inv)};
}

// us of a workgroup over n tiles; load: the share of the CUs that are busy.
// Measured at Q = 1 .. 300, H = 32 .. 256, S = 64 .. 2048, every split count:
// the first tile (page table, q) and a slope, which rises where the
// workgroups share the memory (32 heads, S=2048 Q=1: 59.5, S=600 on 256 CUs: 28.5).
static float split_us(int hg, int n, float load) {
    if (hg == 32 && n > 3 && n * kT32 <= SplitGeom<2, 2>::CHUNK) return 8.8f + (0.8f + 0.24f * load) * n;
    if (hg == 32) return 7.3f + (n > 3 ? 1.5f : 1.3f) * std::max(n, 2);  // (the first two tiles load together)
    if (hg == 64) return 8.3f + 1.58f * n;
    if (hg == 96) return 11.0f + 1.5f * n;
    return 8.4f + (1.8f + 0.5f * load) * n;
}

// Heads per workgroup, splits per query and the bytes of the splits'
// partials.  Head groups of 128 (H a multiple of 128): enough workgroups to
// cover the chip (256 CUs), at most 2048 tokens per split, at least 32.  Small
// groups of 32, 64 or 96 heads (S <= 4096): any split that fits the CUs at
// once, more than one only with scratch.  The cheapest by a model
// fitted to measured calls (us): workgroups run in rounds of 256, a merge takes
// 3 + 0.1 per split and moves its partials at 5.3 MB per us (the 128-head
// merge 4 + 0.5, four splits a round trip, and 16 MB per us of bf16).
// So few queries take many splits of small groups (S=2000 Q=4 H=64: 61 us in one
// split of 32 heads, 19 in 16; S=2048 Q=1 H=128: 48 us in 64 splits of 128 heads,
// 17 so), short selections one split of small groups (S=64 Q=64 H=128: 20 ->
// 10; S=512 Q=64 H=96: 24, 31 in 3 splits of 96), large batches 128 heads.
DsaPlan dsa_paged_plan(int Q, int H, int S, bool scratch) {
    DsaPlan best = {0, 1, 0};
    if (Q < 1 || H < 32 || H % 32 != 0 || S < 1) return best;
    const int tiles = (S + kT32 - 1) / kT32;
    float best_us = 0.0f;
    int full = 0;  // splits of the 128-head form
    auto estimate = [&](int hg, int ns) {
        const long wgs = (long)Q * (H / hg) * ns;
        const float rounds = (float)((wgs + 255) / 256), load = std::min(1.0f, wgs / 256.0f);
        float us = rounds * split_us(hg, (tiles + ns - 1) / ns, load);
        if (hg == 128) us += 4.0f + 0.5f * ns + 2.0f * ns * Q * H * (kDc * 2) / 16e6f;
        else if (ns > 1) us += 3.0f + 0.1f * ns + 2.0f * ns * Q * H * (kDc * 4) / 5.3e6f;
        return us;
    };
    if (H % 128 == 0) {
        const long wg = (long)Q * (H / 128);
        full = (int)std::min<long>((256 + wg - 1) / wg, tiles);
        full = std::max(full, (S + SplitGeom<8, 1>::CHUNK - 1) / SplitGeom<8, 1>::CHUNK);
        best = {128, full, 0};
        best_us = estimate(128, full);
    }
    for (int hg = 32; hg <= 96 && (S <= kMaxS || best.hg == 0); hg += 32) {
        if (H % hg || (hg == 96 && H % 128 == 0)) continue;  // (96: no 64-bit form)
        const long wg = (long)Q * (H / hg);
        const int most = scratch ? (int)std::max(1L, std::min({256 / wg, (long)tiles, 64L})) : 1;
        for (int ns = 1; ns <= most; ns++) {
            const float us = estimate(hg, ns);
            if (best_us == 0.0f || us < best_us) best = {hg, ns, 0}, best_us = us;
        }
    }
    auto bytes = [](size_t rows, int es) { return align_up(rows * kDc * es, 256) + align_up(rows * 8, 256); };
    if (H % 128 == 0)
        // The same bytes whatever form runs: the 128-head form's, and at least
        // what any small groups' splits take (64 heads, 256 workgroups).  The
        // buffer then grows only where the 128-head form needs more: a buffer
        // that a call took for granted in a captured graph is not freed by a
        // smaller call after it.
        best.bytes = std::max(bytes((size_t)Q * full * H, 2), bytes(256 * 64, 4));
    else if (best.ns > 1)
        best.bytes = bytes((size_t)Q * best.ns * H, 4);
    return best;
}

int launch_dsa_bf16_paged(const uint16_t* qn, const uint16_t* qp, const uint16_t* cache,
                          long cache_tokens, const int* page_table, const int* logical,
                          uint16_t* out, int Q, int H, int Dc, int Dp, int S, int page,
                          int pages_per_seq, const DsaPlan& plan, void* scratch, hipStream_t st) {
    AMDMOE_CHECK_ARG(Dc == kDc && Dp == kDp, "dsa_decode_bf16_paged: needs Dc=512, Dp=64 (got %d, %d)", Dc, Dp);
    AMDMOE_CHECK_ARG(H % 32 == 0 && H > 0, "dsa_decode_bf16_paged: H=%d not a multiple of 32", H);
    // 128-head groups take any S up to kMaxSplitS in more splits; the smaller
    // ones may have to take a query's positions in one
    AMDMOE_CHECK_ARG(S >= 1 && S <= (H % 128 == 0 ? kMaxSplitS : kMaxS),
                     "dsa_decode_bf16_paged: S=%d outside [1, %d] for H=%d", S,
                     H % 128 == 0 ? kMaxSplitS : kMaxS, H);
    AMDMOE_CHECK_ARG(page >= 1 && pages_per_seq >= 1, "dsa_decode_bf16_paged: bad paging");
    // caches beyond 4 GiB: the wide kernels address them with 64-bit pointers
    AMDMOE_CHECK_ARG(cache_tokens >= 1 && (cache_tokens * kRowBytes <= kMaxCacheBytes || H % 128 == 0),
                     "dsa_decode_bf16_paged: cache of %ld tokens outside (0, 4 GiB) (larger caches need H a "
                     "multiple of 128)", cache_tokens);
    const bool wide = cache_tokens * kRowBytes > kMaxCacheBytes;
    if (Q == 0) return AMDMOE_OK;
    const float scale_log2 = 1.0f / sqrtf((float)(Dc + Dp)) * 1.4426950408889634f;
    const int hg = plan.hg, ns = plan.ns;
    AMDMOE_CHECK_ARG(hg >= 32 && H % hg == 0 && (plan.bytes == 0 || scratch != nullptr),
                     "dsa_decode_bf16_paged: no scratch for %zu bytes", plan.bytes);
    const int chunk = (int)ceil_div(ceil_div(S, ns), kT32) * kT32;
    const long grid = ceil_div((long)Q * (H / hg) * ns, 8) * 8;  // padded for the XCD dealing
    AMDMOE_CHECK_ARG(grid < (1L << 31), "dsa_decode_bf16_paged: grid too large");
    float* part_ml = plan.bytes ? (float*)((uint8_t*)scratch + align_up((size_t)Q * ns * H * kDc * (hg == 128 ? 2 : 4), 256))
                               : nullptr;
    // two token groups from four tiles on (Q=64 H=32, us without and with: S=64 9.8
    // and 10.4, S=96 11.1 and 12.0, S=112 12.4 and 12.0, S=224 16.9 and 15.2), up to
    // the positions its LDS has room for beside four stages
    const bool pair = hg == 32 && chunk > 3 * kT32 && chunk <= SplitGeom<2, 2>::CHUNK;
    auto split = hg == 128  ? (wide ? dsa_split_wide_kernel : dsa_split_kernel)
                 : hg == 96 ? dsa_split96_kernel
                 : hg == 64 ? (wide ? dsa_split64_wide_kernel : dsa_split64_kernel)
                 : pair     ? (wide ? dsa_split32x2_wide_kernel : dsa_split32x2_kernel)
                            : (wide ? dsa_split32_wide_kernel : dsa_split32_kernel);
    const int lds = hg == 128  ? SplitGeom<8, 1>::LDS
                    : hg == 96 ? SplitGeom<6, 1>::LDS
                    : hg == 64 ? SplitGeom<4, 1>::LDS
                    : pair     ? SplitGeom<2, 2>::LDS
                               : SplitGeom<2, 1>::LDS;
    const int rc = ensure_dynamic_lds((const void*)split, lds);
    if (rc != AMDMOE_OK) return rc;
    hipLaunchKernelGGL(split, dim3((unsigned)grid), dim3(pair ? 256 : 4 * hg), lds, st, qn, qp, cache,
                       cache_tokens * kRowBytes, page_table, logical, out, scratch, part_ml, Q, H, S, page,
                       pages_per_seq, ns, chunk, scale_log2);
    AMDMOE_LAUNCH_CHECK();
    if (ns == 1 && hg != 128) return AMDMOE_OK;
    if (hg == 128)
        hipLaunchKernelGGL(dsa_merge_kernel, dim3((unsigned)(ceil_div((long)Q * (H / 16), 8) * 8)),
                           dim3(256), 0, st, (const uint16_t*)scratch, (const float*)part_ml, out, Q, H, ns);
    else
        hipLaunchKernelGGL(dsa_merge_f32_kernel, dim3((unsigned)(Q * (H / 16) * 16)), dim3(64), 0, st,
                           (const float*)scratch, (const float*)part_ml, out, H, ns);
    AMDMOE_LAUNCH_CHECK();
    return AMDMOE_OK;
}

}  // namespace amdmoe
