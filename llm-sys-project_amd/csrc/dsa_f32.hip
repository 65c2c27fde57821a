// D1, fp32 entry -- DeepSeek sparse attention (MLA absorbed) over flat
// indices, any H, Dc, Dp, S.
//
// Reference: dsa_forward (kernels/dsa/naive_dsa.cu:435-474), the CPU copy
// tests/test_dsa.cu:23-68:
//   s = (dot(q_nope,K_c[i]) + dot(q_pe,K_p[i])) * (1/sqrt(Dc+Dp))
//   P = softmax_S(s);  out = sum_s P*V[i]
//
// The query's valid indices, in order, are cut into chunks of f32_chunk(n)
// positions (n: their count).  One workgroup takes 16 heads of a query over
// a chunk, both products on the fp32 matrix cores:
//   S^T (16 tokens x 16 heads) = K . Q^T   16x16x4 fp32; the operands come
//       straight from memory, 16 bytes per lane (a K row is used once per
//       16 heads, so staging it would only add a pass); the 8 waves split
//       the chunk's token tiles, and the columns when there are fewer tiles
//   p = expf(s - m) 2^-k with the chunk's max m, l = sum p, in LDS; 2^k >= n
//       keeps every partial sum of p V within max |V| (the reference divides
//       before it sums) and divides out exactly at the end
//   O^T (64 dims x 16 heads) += V^T . P^T  16x16x4 fp32; the 8 waves split
//       the 64-dim blocks, and the tokens when there are fewer blocks
// and the chunks' (m, l, O) are folded in order with the usual rescaling:
//   f32_split_kernel + f32_merge_kernel: a workgroup per chunk, the partial
//       O in scratch, for calls too small to fill the chip otherwise
//   f32_loop_kernel: a workgroup walks all chunks of its heads, O
//       accumulating in the output rows; no scratch
// The fold is the same sequence of operations in both, and a chunk depends
// on the query's valid indices alone, so a row's result is bit-identical
// whichever of the two runs, and with or without the invalid indices written
// out.  The smallest calls, and many rows of few heads and columns, run
// f32_row_kernel instead (f32_by_rows: by the call's shape alone), which sums
// in another order.
//
// What bounds it: at Q=8 H=16 Dc=512 Dp=64 S=1024 the call needs 24 MB
// (5 us) and 0.29 GFLOP; it takes 19.5 us, two launches (16 + 4) of a few
// dependent round trips each (indices -> rows -> scores -> V).  One lane per token running
// the reference's sequential dots took 2758 us there: a 64-lane workgroup
// per (query, head) on half the CUs, each lane walking its own K row.
#include "internal.hpp"

#include <float.h>

namespace amdmoe {

// A chunk is 32 positions up to n = 1024, then n/32 (at most 32 chunks) up
// to the 256 whose scores fit LDS beside the rest; a row of at most 128 positions is one
// chunk, because a second launch costs more than the shorter chain saves.
constexpr int kF32One = 128, kF32Min = 32, kF32Max = 256;
constexpr int kF32Waves = 8;
__host__ __device__ inline int f32_chunk(int n) {
    if (n <= kF32One) return kF32One;
    const int c = ((n + 31) / 32 + 15) & ~15;
    return c < kF32Min ? kF32Min : (c > kF32Max ? kF32Max : c);
}
// the most chunks any count of valid positions up to S can have
static int f32_max_chunks(int S) {
    if (S <= kF32One) return 1;
    return std::max(std::min(32, (S + kF32Min - 1) / kF32Min), (S + kF32Max - 1) / kF32Max);
}

struct DsaF32Args {
    const float *qn, *qp, *kc, *kp, *v;
    const int* idx;
    float* out;
    int H, Dc, Dp, S;
    long N;
    int q0;            // split: the first query of this launch
    int nc;            // split: chunk slots per (query, head tile); loop: whether O is in LDS
    float* part_o;     // [query - q0][head tile][chunk][16][Dc]
    float2* part_ml;   // [query - q0][head tile][chunk][16]; l < 0: no such chunk
};

// 4 elements of a row from column k, zeros past D or where !ok.  VEC: rows
// are 16-byte aligned and D is a multiple of 4; the load is unconditional
// (at column 0 where it does not count), so a batch of them stays in flight.
template <bool VEC>
__device__ __forceinline__ f32x4 row4(const float* __restrict__ row, int k, int D, bool ok) {
    f32x4 r = {0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC) {
        const f32x4 t = *(const f32x4*)(row + (k < D ? k : 0));
        if (ok && k < D) r = t;
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float t = row[k + i < D ? k + i : 0];
            if (ok && k + i < D) r[i] = t;
        }
    }
    return r;
}

// pitches of 4 mod 64 floats: the lanes of a P operand (head c, token 4q + g)
// read 64 banks
constexpr int kPPitch = kF32Max + 4, kSPitch = 68;
struct DsaF32Lds {
    int rows[2][kF32Max];                    // cache rows of the chunk (loop: and of the next)
    float p[16 * kPPitch];                   // scores, then probabilities: [head][token]
    float part[kF32Waves * 16 * kSPitch];    // column parts of S^T, then token parts of O^T
    float m[16], l[16];
    int cnt[kF32Waves];
};

// The cache rows of valid positions [c0, c0 + cap) of a query, in order,
// into rows; returns the query's number of valid positions.  Wave w counts
// the indices of its eighth of the list, then places those of the window.
// FIRST: n is not known yet; c0 is a chunk number and cap its chunk's length.
// Each wave's first kKeep * 64 indices stay in registers between the two
// passes (all of them up to S = 2048: one round trip instead of two).
// The cursor is a wave's first group of 64 indices not placed in full, the
// number of valid positions before it, and its indices, loaded ahead: the next
// window goes on there, so walking all windows in turn reads the list once (read
// from the start for every chunk, Q=260 H=16 Dc=64 S=32768 took 5084 us, now 2811).  The
// caller's barrier follows.
struct F32Cursor {
    int s, base, r;
};
template <bool FIRST>
__device__ __forceinline__ int f32_rows(const DsaF32Args& a, DsaF32Lds& L, int* __restrict__ rows,
                                        const int* __restrict__ ir, int n, int c0, int cap, F32Cursor& cur) {
    constexpr int kKeep = 4;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int seg = ((a.S + kF32Waves * 64 - 1) / (kF32Waves * 64)) * 64;
    const int s0 = min(a.S, wave * seg), s1 = min(a.S, s0 + seg);
    auto index = [&](int s) __attribute__((always_inline)) -> int {  // -1: no valid position
        const int r = s < s1 ? ir[s] : -1;
        return r >= 0 && r < a.N ? r : -1;
    };
    // the group at s, base valid positions before it; the next one is r2
    int s = cur.s, base = cur.base;
    auto place = [&](int r, int r2) __attribute__((always_inline)) {
        const unsigned long long mk = __ballot(r >= 0);
        const int at = base + __popcll(mk & ((1ull << lane) - 1)) - c0;
        if (r >= 0 && at >= 0 && at < cap) rows[at] = r;
        base += __popcll(mk);
        s += 64;
        if (base <= c0 + cap) cur = {s, base, r2};
    };
    int r = cur.r;
    if constexpr (FIRST) {
        int keep[kKeep];
#pragma unroll
        for (int k = 0; k < kKeep; k++) keep[k] = index(s0 + 64 * k + lane);
        int c = 0;
#pragma unroll
        for (int k = 0; k < kKeep; k++) c += __popcll(__ballot(keep[k] >= 0));
        for (s = s0 + 64 * kKeep; s < s1; s += 64) c += __popcll(__ballot(index(s + lane) >= 0));
        if (lane == 0) L.cnt[wave] = c;
        lds_barrier();
        n = 0;
        for (int w = 0; w < kF32Waves; w++) n += L.cnt[w];
        cap = f32_chunk(n);
        c0 *= cap;
        s = s0;
        base = 0;
        for (int w = 0; w < wave; w++) base += L.cnt[w];
        cur = {s, base, keep[0]};
        if (base + c <= c0) return n;  // (a wave whose indices all lie before the window places none)
        r = index(s0 + 64 * kKeep + lane);
#pragma unroll
        for (int k = 0; k < kKeep; k++) place(keep[k], k + 1 < kKeep ? keep[k + 1] : r);
    }
    while (s < s1 && base < c0 + cap) {
        const int r2 = index(s + 64 + lane);
        place(r, r2);
        r = r2;
    }
    return n;
}

// How the 8 waves split O^T of a chunk: 64-dim block first + k * step, token
// groups (of 4) [qa, qb); 1 << ts token parts where there are fewer blocks.
struct F32Pv {
    int nb, ts, b, step, qa, qb;
};
__device__ __forceinline__ F32Pv f32_pv_split(int Dc, int len, int wave) {
    F32Pv w;
    w.nb = (Dc + 63) >> 6;
    w.ts = w.nb > 4 ? 0 : w.nb > 2 ? 1 : w.nb > 1 ? 2 : 3;
    const int nq = (len + 3) >> 2, per = (nq + (1 << w.ts) - 1) >> w.ts;
    w.qa = (wave & ((1 << w.ts) - 1)) * per;
    w.qb = min(nq, w.qa + per);
    w.b = wave >> w.ts;
    w.step = kF32Waves >> w.ts;
    return w;
}
constexpr int kPvB = 8;  // token groups whose V loads are in flight together
template <bool VEC>
__device__ __forceinline__ void f32_pv_load(const DsaF32Args& a, const int* rows, const F32Pv& w, int b,
                                            int q, int len, f32x4 (&vv)[kPvB]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < kPvB; j++) {
        const int tok = 4 * (q + j) + (lane >> 4);
        const bool ok = q + j < w.qb && tok < len;
        const long row = rows[ok ? tok : 0];
        vv[j] = row4<VEC>(a.v + row * a.Dc, 64 * b + 4 * (lane & 15), a.Dc, ok && b < w.nb);
    }
    __builtin_amdgcn_sched_barrier(0);
}

// (m, l) of a chunk of len (1 .. kF32Max) of the query's n positions, its
// rows in rows: leaves p = expf(s - m) 2^-k in L.p, zero past len.  The first V loads
// of f32_pv go out (into vv) once the K loads have, under the softmax.
template <bool VEC>
__device__ __forceinline__ void f32_scores(const DsaF32Args& a, DsaF32Lds& L, const int* rows, int qi, int h0, int n, int len,
                                           float scale, f32x4 (&vv)[kPvB]) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int nt = (len + 15) >> 4;
    const int ks = nt > 4 ? 0 : nt > 2 ? 1 : nt > 1 ? 2 : 3, kp = 1 << ks;  // column parts
    const int nsc = (a.Dc + 15) >> 4, ns = nsc + ((a.Dp + 15) >> 4);        // 16-column steps
    const int per = (ns + kp - 1) >> ks;
    const int part = wave & (kp - 1);
    const int sa = part * per, sb = min(ns, sa + per);
    const bool hok = h0 + c < a.H;
    const size_t qrow = (size_t)qi * a.H + (hok ? h0 + c : h0);
    const float* qn = a.qn + qrow * a.Dc;
    const float* qp = a.qp + qrow * a.Dp;
    for (int t = wave >> ks; t < nt; t += kF32Waves >> ks) {
        const int tok = 16 * t + c;
        const bool tok_ok = tok < len;
        const long row = rows[tok_ok ? tok : 0];
        const float* kc = a.kc + row * a.Dc;
        const float* kq = a.kp + row * a.Dp;
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        auto steps = [&](auto bc) __attribute__((always_inline)) {
            constexpr int kB = decltype(bc)::value;  // steps whose loads are in flight together
            for (int s = sa; s < sb; s += kB) {
                f32x4 kv[kB], qv[kB];
#pragma unroll
                for (int j = 0; j < kB; j++) {
                    const bool live = s + j < sb;                // uniform
                    const int st = live ? s + j : sa;
                    const bool first = st < nsc;                 // uniform
                    const int k = 16 * (first ? st : st - nsc) + 4 * g;
                    kv[j] = row4<VEC>(first ? kc : kq, k, first ? a.Dc : a.Dp, tok_ok && live);
                    qv[j] = row4<VEC>(first ? qn : qp, k, first ? a.Dc : a.Dp, hok && live);
                }
#pragma unroll
                for (int j = 0; j < kB; j++)
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[i & 1] = mfma_f32(kv[j][i], qv[j][i], acc[i & 1]);
            }
        };
        // (a batch loads all of its steps, live or not)
        if (VEC && per <= 3) steps(std::integral_constant<int, 3>());
        else steps(std::integral_constant<int, VEC ? 9 : 4>());
        // lane: head c, tokens 16t + 4g + i; kp > 1: at most 4 tiles
        float* dst = kp == 1 ? L.p + c * kPPitch : L.part + (part * 16 + c) * kSPitch;
        *(f32x4*)(dst + 16 * t + 4 * g) = acc[0] + acc[1];
    }
    {
        const F32Pv w = f32_pv_split(a.Dc, len, wave);
        f32_pv_load<VEC>(a, rows, w, w.b, w.qa, len, vv);
    }
    lds_barrier();
    // half a wave per head: lane j takes tokens j, j + 32, ...
    const int hd = 2 * wave + (lane >> 5), j = lane & 31;
    float* ph = L.p + hd * kPPitch;
    float mx = -INFINITY;
#pragma unroll 1
    for (int t = j; t < 16 * nt; t += 32) {
        float s = kp == 1 ? ph[t] : 0.0f;
        if (kp > 1)
            for (int k = 0; k < kp; k++) s += L.part[(k * 16 + hd) * kSPitch + t];
        s = t < len ? s * scale : -INFINITY;
        ph[t] = s;
        mx = fmaxf(mx, s);
    }
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
    const float mu = mx == -INFINITY ? 0.0f : mx;  // every score -inf: p = 0
    const float pn = __int_as_float((95 + __clz(n - 1)) << 23);  // 2^-k, k = 32 - clz(n - 1)
    float sum = 0.0f;
#pragma unroll 1
    for (int t = j; t < 16 * nt; t += 32) {
        const float p = t < len ? expf(ph[t] - mu) * pn : 0.0f;
        ph[t] = p;
        sum += p;
    }
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) sum += __shfl_xor(sum, o, kWave);
    if (j == 0) L.m[hd] = mx, L.l[hd] = sum;
    lds_barrier();
}

// O of the chunk, 64 dims at a time: store(head, dim, 4 values).
template <bool VEC, typename Store>
__device__ __forceinline__ void f32_pv(const DsaF32Args& a, DsaF32Lds& L, const int* rows, int len, f32x4 (&vv)[kPvB],
                                       const Store& store) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const F32Pv w = f32_pv_split(a.Dc, len, wave);
    const int nb = w.nb, tp = 1 << w.ts;
    for (int b = w.b; b - w.b < nb; b += w.step) {
        f32x4 acc[4];
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
        for (int q = w.qa; q < w.qb && b < nb; q += kPvB) {
            if (q > w.qa || b > w.b) f32_pv_load<VEC>(a, rows, w, b, q, len, vv);
#pragma unroll
            for (int j = 0; j < kPvB; j++) {
                const int tok = 4 * (q + j) + g;
                const float p = q + j < w.qb && tok < len ? L.p[c * kPPitch + tok] : 0.0f;
#pragma unroll
                for (int i = 0; i < 4; i++) acc[i] = mfma_f32(vv[j][i], p, acc[i]);
            }
        }
        // acc[i][j], lane (head c, group g): dim 64b + 16g + 4j + i
        if (tp > 1) {  // (then there is one round; parts at kSPitch: at 64 all heads' stores share their banks)
            lds_barrier();
            if (b < nb)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    *(f32x4*)(L.part + (wave * 16 + c) * kSPitch + 16 * g + 4 * j) =
                        (f32x4){acc[0][j], acc[1][j], acc[2][j], acc[3][j]};
            lds_barrier();
            for (int e = tid; e < nb * 256; e += 64 * kF32Waves) {  // 4 dims of a head
                const int bb = e >> 8, hd = (e >> 4) & 15, dd = 4 * (e & 15);
                f32x4 o = {0.f, 0.f, 0.f, 0.f};
                for (int k = 0; k < tp; k++) o += *(const f32x4*)(L.part + ((bb * tp + k) * 16 + hd) * kSPitch + dd);
                store(hd, 64 * bb + dd, o);
            }
        } else if (b < nb) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                store(c, 64 * b + 16 * g + 4 * j, (f32x4){acc[0][j], acc[1][j], acc[2][j], acc[3][j]});
        }
    }
}

// One step of the fold: (m, l, O) so far and a chunk's (mj, lj, Oj) become
// O * c0 + Oj * c1.  A chunk without a finite score has weight 0 (its NaNs,
// if any, still reach the sums, as in the reference).
struct F32Fold {
    float c0, c1;
};
__device__ __forceinline__ F32Fold f32_fold(float& m, float& l, float mj, float lj) {
    const float mn = fmaxf(m, mj);
    F32Fold f;
    f.c0 = m == -INFINITY ? 0.0f : expf(m - mn);
    f.c1 = mj == -INFINITY ? 0.0f : expf(mj - mn);
    l = fmaf(l, f.c0, mul_rn(lj, f.c1));
    m = mn;
    return f;
}
__device__ __forceinline__ float f32_fold_o(const F32Fold& f, float o, float oj) {
    return fmaf(o, f.c0, mul_rn(oj, f.c1));
}
__device__ __forceinline__ float f32_inv(float m, float l) { return m == -INFINITY ? 0.0f : __fdiv_rn(1.0f, l); }

template <bool VEC>
__device__ __forceinline__ void store4(float* __restrict__ row, int d, int D, f32x4 v) {
    if constexpr (VEC) {
        if (d < D) *(f32x4*)(row + d) = v;
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (d + i < D) row[d + i] = v[i];
    }
}

template <bool VEC>
__global__ __launch_bounds__(512) void f32_split_kernel(DsaF32Args a) {
    __shared__ DsaF32Lds L;
    const int ht = (a.H + 15) >> 4;
    const int sp = blockIdx.x % a.nc, qt = blockIdx.x / a.nc;
    const int qi = a.q0 + qt / ht, h0 = 16 * (qt % ht);
    F32Cursor cur = {0, 0, -1};
    const int n = f32_rows<true>(a, L, L.rows[0], a.idx + (size_t)qi * a.S, 0, sp, 0, cur);
    const int chunk = f32_chunk(n), c0 = sp * chunk;
    const size_t slot = (size_t)blockIdx.x * 16;
    if (c0 >= n) {
        if (threadIdx.x < 16) a.part_ml[slot + threadIdx.x] = make_float2(-INFINITY, -1.0f);
        return;
    }
    lds_barrier();
    const int len = min(chunk, n - c0);
    f32x4 vv[kPvB];
    f32_scores<VEC>(a, L, L.rows[0], qi, h0, n, len, 1.0f / sqrtf((float)(a.Dc + a.Dp)), vv);
    if (threadIdx.x < 16) a.part_ml[slot + threadIdx.x] = make_float2(L.m[threadIdx.x], L.l[threadIdx.x]);
    f32_pv<VEC>(a, L, L.rows[0], len, vv, [&](int hd, int d, f32x4 o) __attribute__((always_inline)) {
        if (h0 + hd < a.H) store4<VEC>(a.part_o + (slot + hd) * a.Dc, d, a.Dc, o);
    });
}

// A wave per (query, head, 64 dims): the fold over the chunks, 32 at a time
// with all their loads in flight; lanes 16u .. 16u + 15 hold chunks 8u ..
// 8u + 7 and the four groups fold in turn.  Lane (u, j) works out the factors
// of chunk 8u + j (a running maximum is exact in any order, so they are those
// of the sequential fold).  Short code matters as much as the loads: with
// the 32 folds unrolled in one wave of 256 dims the kernel took 15 us at Q=8
// H=16 S=1024, most of it fetching instructions that run once.
template <bool VEC>
__global__ __launch_bounds__(64) void f32_merge_kernel(DsaF32Args a) {
    const int nd = (a.Dc + 63) >> 6;
    const int lane = threadIdx.x, u = lane >> 4;
    const int qh = blockIdx.x / nd;
    const int d = 64 * (blockIdx.x - qh * nd) + 4 * (lane & 15);
    const int ql = qh / a.H, hd = qh - ql * a.H;
    const int ht = (a.H + 15) >> 4;
    const size_t slot0 = ((size_t)ql * ht + (hd >> 4)) * a.nc * 16 + (hd & 15);
    float m = -INFINITY;
    float o[5] = {0.f, 0.f, 0.f, 0.f, 0.f};  // 4 dims and l
    for (int j0 = 0; j0 < a.nc; j0 += 32) {
        const int mine = j0 + 8 * u + (lane & 7);
        float2 ml = a.part_ml[slot0 + (size_t)min(mine, a.nc - 1) * 16];
        f32x4 ov[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            ov[j] = row4<VEC>(a.part_o + (slot0 + (size_t)min(j0 + 8 * u + j, a.nc - 1) * 16) * a.Dc, d, a.Dc, true);
        __builtin_amdgcn_sched_barrier(0);
        if (mine >= a.nc) ml = make_float2(-INFINITY, -1.0f);  // no such chunk
        // the maximum up to and before this lane's chunk (lanes 8 .. 15 of a group repeat 0 .. 7)
        float incl = ml.x;
#pragma unroll 1
        for (int s = 1; s < 8; s <<= 1) {
            const float up = __shfl_up(incl, s, 8);
            if ((lane & 7) >= s) incl = fmaxf(incl, up);
        }
        float top = m;  // over the groups before this lane's
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float t = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(incl), 16 * g + 7));
            if (g < u) top = fmaxf(top, t);
            m = fmaxf(m, t);
        }
        float mm = __shfl_up(incl, 1, 8);
        mm = (lane & 7) == 0 ? top : fmaxf(top, mm);
        float ll = 0.0f;
        const F32Fold f = f32_fold(mm, ll, ml.x, ml.y);
        float c0[8], c1[8], lj[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            c0[j] = __shfl(f.c0, j, 16);
            c1[j] = __shfl(f.c1, j, 16);
            lj[j] = __shfl(ml.y, j, 16);
        }
#pragma unroll 1
        for (int g = 0; g < 4; g++) {  // group g's lanes continue the fold, then hand it on
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const F32Fold fj = {c0[j], c1[j]};
                const bool there = lj[j] >= 0.0f || lj[j] != lj[j];
#pragma unroll
                for (int i = 0; i < 4; i++) o[i] = there ? f32_fold_o(fj, o[i], ov[j][i]) : o[i];
                o[4] = there ? f32_fold_o(fj, o[4], lj[j]) : o[4];
            }
#pragma unroll
            for (int i = 0; i < 5; i++) o[i] = __shfl(o[i], 16 * g + (lane & 15), kWave);
        }
    }
    if (u) return;
    const float inv = f32_inv(m, o[4]);
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = m == -INFINITY ? 0.0f : mul_rn(o[i], inv);
    store4<VEC>(a.out + ((size_t)(a.q0 + ql) * a.H + hd) * a.Dc, d, a.Dc, r);
}

// The same fold by one workgroup: a thread has the same dims of the same head in
// every chunk, so it keeps that head's (m, l) and O, in LDS where there is room
// (nc = 1: up to 320 columns for two workgroups on a CU, 512 for one), else in
// the output rows.
// The next chunk's rows are placed before the barrier that ends a chunk, from
// indices loaded a chunk earlier.  A chunk is a chain of latencies: Q=4 H=8 Dc=32
// S=1024 (32 chunks) in one launch took 278 us with O in the output rows, the fold
// between two barriers of its own and bank conflicts in the token parts (21000
// cycles a chunk, 4300 of them those stores, 6600 rows and scores), 178 so.
constexpr int kLoopDc2 = 320, kLoopDc1 = 512;
__host__ __device__ inline int f32_loop_pitch(int Dc) { return ((Dc + 63) & ~63) + 4; }
template <bool VEC>
__global__ __launch_bounds__(512, 4) void f32_loop_kernel(DsaF32Args a) {
    __shared__ DsaF32Lds L;
    extern __shared__ __attribute__((aligned(16))) float s_o[];  // [head][f32_loop_pitch(Dc)]
    const int ht = (a.H + 15) >> 4;
    const int qi = blockIdx.x / ht, h0 = 16 * (blockIdx.x % ht);
    const int tid = threadIdx.x;
    const int* ir = a.idx + (size_t)qi * a.S;
    float* orow = a.out + ((size_t)qi * a.H + h0) * a.Dc;
    const float scale = 1.0f / sqrtf((float)(a.Dc + a.Dp));
    const bool lds_o = a.nc != 0;
    const int pitch = f32_loop_pitch(a.Dc);
    const int hd_own = a.Dc <= 256 ? (tid >> 4) & 15 : tid & 15;  // the head f32_pv gives this thread
    float m = -INFINITY, l = 0.0f;                                // of that head
    F32Cursor cur = {0, 0, -1};
    const int n = f32_rows<true>(a, L, L.rows[0], ir, 0, 0, 0, cur);
    if (n == 0) {  // no valid index
        for (int i = tid; i < 16 * a.Dc; i += 512)
            if (h0 + i / a.Dc < a.H) orow[i] = 0.0f;
        return;
    }
    const int chunk = f32_chunk(n);
    int buf = 0;
    for (int c0 = 0; c0 < n; c0 += chunk, buf ^= 1) {
        if (c0) f32_rows<false>(a, L, L.rows[buf], ir, n, c0, chunk, cur);
        lds_barrier();  // the rows are there, the last chunk's probabilities have been read
        const int len = min(chunk, n - c0);
        f32x4 vv[kPvB];
        f32_scores<VEC>(a, L, L.rows[buf], qi, h0, n, len, scale, vv);
        const F32Fold f = f32_fold(m, l, L.m[hd_own], L.l[hd_own]);
        const float inv = f32_inv(m, l);
        const bool last = c0 + chunk >= n;
        f32_pv<VEC>(a, L, L.rows[buf], len, vv, [&](int hd, int d, f32x4 oj) __attribute__((always_inline)) {
            if (h0 + hd >= a.H) return;
            float* row = orow + (size_t)hd * a.Dc;
            float* so = s_o + hd * pitch + d;
            f32x4 o = {0.f, 0.f, 0.f, 0.f};
            if (c0) {
                if (lds_o) o = *(const f32x4*)so;
                else o = row4<VEC>(row, d, a.Dc, true);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                o[i] = f32_fold_o(f, o[i], oj[i]);
                if (last) o[i] = m == -INFINITY ? 0.0f : mul_rn(o[i], inv);
            }
            if (lds_o && !last) *(f32x4*)so = o;
            else store4<VEC>(row, d, a.Dc, o);
        });
    }
}

// A wave per (query, head), lane j with positions j, j + 64, ...: four sums over
// the columns of its rows, then lanes own output columns.  For the smallest
// calls, where the kernels above take 9 us however little there is to do (512
// threads, six barriers), and for many rows of few heads and columns, where they
// run whole chunks for one or two of a tile's 16 heads.
template <bool VEC>
__global__ __launch_bounds__(64) void f32_row_kernel(DsaF32Args a) {
    extern __shared__ float s_p[];  // [S] scores, then probabilities
    int* s_row = (int*)(s_p + a.S);
    const int qh = blockIdx.x, qi = qh / a.H, lane = threadIdx.x;
    const float *qn = a.qn + (size_t)qh * a.Dc, *qp = a.qp + (size_t)qh * a.Dp;
    const int* ir = a.idx + (size_t)qi * a.S;
    const float scale = 1.0f / sqrtf((float)(a.Dc + a.Dp));
    float mx = -INFINITY;
    for (int s = lane; s < a.S; s += 64) {
        const int r = ir[s];
        const bool ok = r >= 0 && r < a.N;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        auto dot = [&](const float* q, const float* k, int D) __attribute__((always_inline)) {
#pragma unroll 4
            for (int d = 0; d < D; d += 4) {
                const f32x4 kv = row4<VEC>(k, d, D, true), qv = row4<VEC>(q, d, D, true);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[i] = fmaf(kv[i], qv[i], acc[i]);
            }
        };
        float p = -INFINITY;
        if (ok) {
            dot(qn, a.kc + (size_t)r * a.Dc, a.Dc);
            dot(qp, a.kp + (size_t)r * a.Dp, a.Dp);
            p = ((acc[0] + acc[1]) + (acc[2] + acc[3])) * scale;
        }
        mx = fmaxf(mx, p);
        s_p[s] = p;
        s_row[s] = ok ? r : -1;
    }
    mx = wave_max(mx);
    float* out = a.out + (size_t)qh * a.Dc;
    if (mx == -INFINITY) {  // no score above -inf
        for (int d = lane; d < a.Dc; d += 64) out[d] = 0.0f;
        return;
    }
    float tot = 0.0f;
    for (int s = lane; s < a.S; s += 64) tot += s_p[s] = expf(s_p[s] - mx);
    tot = wave_sum(tot);
    for (int s = lane; s < a.S; s += 64) s_p[s] = __fdiv_rn(s_p[s], tot);
    __syncthreads();
    for (int d = lane; d < a.Dc; d += 64) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
        for (int s = 0; s < a.S; s += 4) {
            float v[4], p[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int t = min(s + i, a.S - 1), r = s_row[t];
                const bool ok = s + i < a.S && r >= 0;
                const float x = a.v[(size_t)max(r, 0) * a.Dc + d];
                v[i] = ok ? x : 0.0f;
                p[i] = ok ? s_p[t] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i] = fmaf(p[i], v[i], acc[i]);
        }
        out[d] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    }
}

// ---------------------------------------------------------------- launch
static long f32_head_tiles(int Q, int H) { return (long)Q * ((H + 15) / 16); }
// Is f32_row_kernel the faster one?  Both times in ns, fitted to 1000 calls (Q = 1
// .. 2500, H = 1 .. 16, Dc = 8 .. 512, S = 1 .. 1024): a wave's chain over its
// positions and their traffic, against one chunk (8 us, in rounds of 512
// workgroups) or a full chip's walks (5.5 us per chunk, 7.6 with two workgroups
// on a CU); a row of several chunks on few CUs is always split.  Tiles and rows,
// us: Q=1 H=1 Dc=32 Dp=4 S=1 8.0 and 3.8, S=64 9.1 and 9.0; Dc=128 Dp=32 S=16 9.1 and
// 7.2, S=32 9.2 and 9.9; Q=1000 H=1 Dc=32 S=1024 486 and 116; Q=1000 H=4 Dc=128 513
// and 506; Q=256 H=16 Dc=64 185 and 253.  It depends on the shape alone, so eager
// and captured calls agree.
static bool f32_by_rows(int Q, int H, int Dc, int Dp, int S) {
    const long tiles = f32_head_tiles(Q, H), rows = (long)Q * H, D = (long)Dc + Dp;
    if (S > 2048 || (S > kF32One && tiles < 256)) return false;
    const long rounds = (tiles + 511) / 512;
    const float row = 3200.0f + 13.0f * D + (float)S * ((Dc + 63) / 64) * (82.0f + 0.042f * rows);
    const float tile = S > kF32One      ? 4000.0f + (S + f32_chunk(S) - 1) / f32_chunk(S) * rounds * (tiles <= 256 ? 5500.0f : 7600.0f)
                       : tiles <= 256 ? 8000.0f + 3.6f * D + 12.0f * S
                                      : 4000.0f + rounds * (8000.0f + 30.0f * S);
    return row < 0.95f * tile;
}
// The split form runs where a workgroup per (query, 16 heads) leaves CUs
// idle: fewer than 256 of them, and rows of more than one chunk.
static size_t f32_query_bytes(int H, int Dc, int S) {  // partials of one query
    const size_t slots = (size_t)((H + 15) / 16) * f32_max_chunks(S) * 16;
    return slots * Dc * 4 + slots * 8;
}
constexpr size_t kF32Pad = 512;                      // the (m, l) pairs' alignment
constexpr size_t kF32Scratch = (64u << 20) - kF32Pad;  // queries are taken in groups whose partials fit this

size_t dsa_f32_scratch_bytes(int Q, int H, int Dc, int S) {
    if (Q < 1 || H < 1 || f32_max_chunks(S) == 1 || f32_head_tiles(Q, H) >= 256) return 0;
    const size_t one = f32_query_bytes(H, Dc, S);
    const size_t group = std::max<size_t>(1, std::min<size_t>(Q, kF32Scratch / one));
    return one > kF32Scratch ? 0 : group * one + kF32Pad;
}

template <bool VEC>
static int launch_f32(DsaF32Args a, int Q, void* scratch, size_t scratch_bytes, hipStream_t st) {
    const long tiles = f32_head_tiles(Q, a.H);
    if (!scratch) {
        AMDMOE_CHECK_ARG(tiles < (1L << 31), "dsa_forward: grid too large");
        a.nc = a.Dc <= (tiles <= 256 ? kLoopDc1 : kLoopDc2);
        const int lds = a.nc ? 16 * f32_loop_pitch(a.Dc) * 4 : 0;
        const int rc = ensure_dynamic_lds((const void*)f32_loop_kernel<VEC>, 16 * f32_loop_pitch(kLoopDc1) * 4);
        if (rc != AMDMOE_OK) return rc;
        hipLaunchKernelGGL(f32_loop_kernel<VEC>, dim3((unsigned)tiles), dim3(512), lds, st, a);
        AMDMOE_LAUNCH_CHECK();
        return AMDMOE_OK;
    }
    const int ht = (a.H + 15) / 16, nd = (a.Dc + 63) / 64;
    a.nc = f32_max_chunks(a.S);
    const int group = (int)std::min<size_t>(Q, (scratch_bytes - kF32Pad) / f32_query_bytes(a.H, a.Dc, a.S));
    AMDMOE_CHECK_ARG(group >= 1, "dsa_forward: scratch of %zu bytes", scratch_bytes);
    const size_t slots = (size_t)group * ht * a.nc * 16;
    a.part_o = (float*)scratch;
    a.part_ml = (float2*)((uint8_t*)scratch + align_up(slots * a.Dc * 4, 256));
    for (int q0 = 0; q0 < Q; q0 += group) {
        a.q0 = q0;
        const unsigned nq = (unsigned)std::min(Q - q0, group);
        hipLaunchKernelGGL(f32_split_kernel<VEC>, dim3(nq * ht * a.nc), dim3(512), 0, st, a);
        AMDMOE_LAUNCH_CHECK();
        hipLaunchKernelGGL(f32_merge_kernel<VEC>, dim3(nq * a.H * nd), dim3(64), 0, st, a);
        AMDMOE_LAUNCH_CHECK();
    }
    return AMDMOE_OK;
}

int launch_dsa_f32(const float* qn, const float* qp, const float* kc, const float* kp,
                   const float* v, const int* idx, float* out, int Q, int H, int Dc, int Dp, int S,
                   int N, void* scratch, size_t scratch_bytes, hipStream_t st) {
    if (Q == 0 || H == 0) return AMDMOE_OK;
    DsaF32Args a{};
    a.qn = qn, a.qp = qp, a.kc = kc, a.kp = kp, a.v = v, a.idx = idx, a.out = out;
    a.H = H, a.Dc = Dc, a.Dp = Dp, a.S = S, a.N = N;
    // 16-byte loads: whole rows of 16 bytes at aligned bases (Dp = 0 reads no q_pe / K_p)
    auto al = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
    const bool vec = Dc % 4 == 0 && Dp % 4 == 0 && al(qn) && al(kc) && al(v) && al(out) &&
                     (Dp == 0 || (al(qp) && al(kp)));
    if (f32_by_rows(Q, H, Dc, Dp, S)) {
        AMDMOE_CHECK_ARG((long)Q * H < (1L << 31), "dsa_forward: grid too large");
        auto kern = vec ? f32_row_kernel<true> : f32_row_kernel<false>;
        hipLaunchKernelGGL(kern, dim3((unsigned)((long)Q * H)), dim3(64), 8 * (size_t)S, st, a);
        AMDMOE_LAUNCH_CHECK();
        return AMDMOE_OK;
    }
    return vec ? launch_f32<true>(a, Q, scratch, scratch_bytes, st)
               : launch_f32<false>(a, Q, scratch, scratch_bytes, st);
}

}  // namespace amdmoe
