// fused_kernels.hip -- one-pass Lloyd step for small k*d on gfx950 (MI355X):
// the E-step (sklearn/cluster/_k_means_lloyd.pyx:196-212) and the
// per-cluster sums and counts of the M-step (:214-218) in one kernel that
// reads X from HBM once per step.
//
//   k_fused     E-step on fp32 MFMA, per-cluster sums by a VALU walker; 8
//               waves per block (d <= 16, data outside the split's range of
//               split_kernels.hip's k_fused3, or the fp32 switch).
//   k_fused_low E-step and sums on the VALU, every wave by itself (d <= 16,
//               few centres or many rows: low_takes).
//
// The fused kernels are used when k <= 64 and d <= 100; X's row stride ld is
// then padded (with zeros) to 4*NQ floats for one of the compiled NQ, so the
// kernels' loops over the row's float4s have no bounds.  The separate assign
// / update kernels cover every other shape.
//
// Built without -amdgpu-mfma-vgpr-form (the register allocator places the
// MFMA accumulators).
#include <math.h>
#include <stdlib.h>

#include "fused_common.h"

namespace skm {

// A block is 8 waves, two per SIMD: MFMA waves 0-3 and walker waves 4-7.
// MFMA wave p and walker wave 4+p form pair p and share one 64-row LDS tile;
// pair p of block b handles tiles t = 4b + p + r*P (P = 4 * blocks) in
// rounds r.  A wave cannot issue VALU work while its own MFMAs run, but the
// other wave on the same SIMD can, so the walker's adds overlap the MFMA
// wave's E-step.  The two waves of a pair hand tiles over through LDS flags;
// there is no block barrier until the end.
//
//   MFMA wave  holds tile t's row in registers (one row per lane) and runs
//              the E-step as k_assign does: x.c on v_mfma_f32_4x4x1_16b_f32
//              (B = this lane's row, A = centres from LDS, lane j = cluster
//              j), ||c||^2 - 2 x.c and the first minimum in the lane.  From
//              chunk K on, each chunk is written to the pair's LDS tile right
//              after its MFMAs (once the walker has read that chunk of tile
//              t - P: it publishes its progress per chunk) and its registers
//              are reloaded with tile t + P, so the HBM reads spread over the
//              E-step.  Chunks [0, K) are held in one
//              of two register sets (by round parity), written out after the
//              argmin and reloaded with tile t + 2P.  Then the tile's rows of
//              each cluster go to LDS as bit masks (an LDS atomic OR of
//              1 << lane into mask[label]; OR does not depend on the order the
//              lanes land in) and the tile is flagged ready.
//   walker     lane j adds the ready tile's rows of cluster j to its running
//              sums of every column, in registers: the lowest WS bits of its
//              mask become LDS row offsets (unused ones point at a row of
//              zeros, so the walk is a fixed sequence), rows past the first
//              WS by a loop; it flags each chunk as soon as its reads are
//              issued.
//
// Rows are added in ascending row order per cluster (the first WS rows after
// the others), tiles in round order, and the four walkers are combined in
// wave order: bitwise reproducible.
// Rows per (cluster, tile) walked without a loop: about the mean 64/k plus
// three standard deviations for balanced clusters.
template <int KG>
__host__ __device__ constexpr int walk_steps()
{
    return KG >= 12 ? 6 : KG >= 8 ? 8 : KG >= 4 ? 12 : 16;
}
// Buffer descriptor over the rows of tile t (none past the last row: loads
// there return 0 without a memory access).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const float* X, long t, long n, int ld)
{
    const long r0 = t * 64;
    const long rows = n - r0 < 64 ? (n - r0 > 0 ? n - r0 : 0) : 64;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(X + (rows > 0 ? r0 * ld : 0)), (short)0,
                                             (int)(rows * ld * 4), 0x00020000);
}
// First minimum of d[0..N) with its index, as a pairwise tree in which the
// lower-index side wins ties -- the same result as scanning j upward with a
// strict '<' from +inf (NaN never wins: leaves are clamped to +inf first).
template <int N>
__device__ __forceinline__ int argmin_tree(float* d)
{
    int ix[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        d[j] = fminf(d[j], INFINITY);
        ix[j] = j;
    }
#pragma unroll
    for (int w = 1; w < N; w *= 2) {
#pragma unroll
        for (int j = 0; j + w < N; j += 2 * w) {
            const bool take = d[j + w] < d[j];
            d[j] = take ? d[j + w] : d[j];
            ix[j] = take ? ix[j + w] : ix[j];
        }
    }
    return ix[0];
}
// The walker wave of a pair: for every round, waits for the tile, then lane j
// adds the tile's rows of cluster j (its mask) to S, publishing its progress
// per chunk; cnt counts the rows.
template <int CPC, int WS, int NQ, int XS>
__device__ __forceinline__ void walk_tiles(float4 (&S)[NQ], int& cnt, int rounds, int lane, int* ready, int* prog,
                                           const unsigned long long* mask, const char* lbase, int toff, int zoff)
{
#pragma unroll
    for (int q = 0; q < NQ; ++q) S[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    cnt = 0;
    for (int r = 0; r < rounds; ++r) {
        wait_flag(ready, r + 1);
        unsigned long long m = lane < CPC ? mask[lane] : 0ull;
        cnt += (int)__popcll(m);
        int ro[WS];
#pragma unroll
        for (int s = 0; s < WS; ++s) {
            const int rr = __ffsll((long long)m) - 1;
            ro[s] = m != 0ull ? toff + rr * XS * 4 : zoff;
            m &= m - 1ull;
        }
        // rows past the first WS (ascending) first, then the first WS: a
        // fixed order either way
        if (__ballot(m != 0ull) != 0ull) {
            while (m != 0ull) {
                const int rr = __ffsll((long long)m) - 1;
                m &= m - 1ull;
                const char* src = lbase + toff + rr * XS * 4;
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    const float4 v = *reinterpret_cast<const float4*>(src + 16 * q);
                    S[q].x += v.x;
                    S[q].y += v.y;
                    S[q].z += v.z;
                    S[q].w += v.w;
                }
            }
        }
        float4 wv[WS];
#pragma unroll
        for (int s = 0; s < WS; ++s) wv[s] = *reinterpret_cast<const float4*>(lbase + ro[s]);
        set_flag(prog, r * NQ + 1);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            float4 wn[WS];
            if (q + 1 < NQ) {
#pragma unroll
                for (int s = 0; s < WS; ++s) wn[s] = *reinterpret_cast<const float4*>(lbase + ro[s] + 16 * (q + 1));
                set_flag(prog, r * NQ + q + 2);  // reads issued: LDS keeps their order
            }
#pragma unroll
            for (int s = 0; s < WS; ++s) {
                S[q].x += wv[s].x;
                S[q].y += wv[s].y;
                S[q].z += wv[s].z;
                S[q].w += wv[s].w;
            }
            if (q + 1 < NQ) {
#pragma unroll
                for (int s = 0; s < WS; ++s) wv[s] = wn[s];
            }
        }
    }
}

// After the tiles: every walker's sums into red = [4][CPC][ld] (over the tile
// area, once every pair is done with it), then the block's partial sums and
// counts, the four walkers combined in wave order.
template <int CPC, int NQ>
__device__ __forceinline__ void publish_sums(const float4 (&S)[NQ], int cnt, float* red, int ld, int pair, int lane,
                                             int (*sCnt)[64])
{
    if (lane < CPC) {
        float* dst = red + (pair * CPC + lane) * ld;
#pragma unroll
        for (int q = 0; q < NQ; ++q) *reinterpret_cast<float4*>(dst + 4 * q) = S[q];
        sCnt[pair][lane] = cnt;
    }
}
template <int KG, int NQ>
__global__ __launch_bounds__(512, 1) void k_fused(FusedArgs a)
{
    const float* __restrict__ X = a.X;
    const long n = a.n;
    const int ld = a.ld;
    const float* __restrict__ C = a.C;
    const int k = a.k;
    int* __restrict__ labels = a.labels;
    float* __restrict__ psum = a.psum;
    int* __restrict__ pcnt = a.pcnt;
    LoopState* st = a.state;
    constexpr int CPC = 4 * KG;
    constexpr int WS = walk_steps<KG>();
    constexpr int XS = fused_stride(NQ);      // ld == 4 * NQ
    constexpr int K = NQ >= 8 ? 3 : NQ / 2;  // chunks computed before the LDS tile is reused
    constexpr int KA = K > 0 ? K : 1;
    constexpr int LB = 8;                     // chunks per burst of HBM loads
    // LDS: centres [CPC x XS] | zero row [XS] | 4 pair tiles [64 x XS]
    extern __shared__ __attribute__((aligned(16))) float lds[];
    __shared__ unsigned long long sMask[4][64];
    __shared__ int sCnt[4][64];
    __shared__ __attribute__((aligned(16))) float sN[CPC];
    __shared__ int sReady[4];  // tiles the MFMA wave has put in LDS
    __shared__ int sProg[4];   // chunks the walker has read: tile * NQ + chunk
    __shared__ int sDone;      // nonzero: the loop has halted, nothing to do
    __shared__ int sChg;       // labels the block's MFMA waves changed
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: keeps descriptors scalar
    const int pair = wave & 3;

    float* sC = lds;
    float* zrow = lds + CPC * XS;
    float* tile = zrow + XS + pair * 64 * XS;
    const int zoff = CPC * XS * 4;  // byte offsets from `lds`
    const int toff = (CPC + 1 + pair * 64) * XS * 4;
    const char* lbase = reinterpret_cast<const char*>(lds);

    const long ntiles = (n + 63) >> 6;
    const long P = (long)gridDim.x * 4;
    const long t0 = (long)blockIdx.x * 4 + pair;
    const int rounds = t0 < ntiles ? (int)((ntiles - t0 + P - 1) / P) : 0;  // this pair's tiles
    const int xoff = lane * ld * 4;  // this lane's row inside a tile of X

    if (wave < 4) {
        // MFMA wave.  Tile t's row: chunks [0, K) in pre (two sets, one per
        // round parity, loaded a round ahead), chunks [K, NQ) in xv.  The
        // first tiles are requested before anything else: their HBM latency
        // overlaps the walkers' set-up.
        float4 preA[KA], preB[KA], xv[NQ - K];
        const __amdgpu_buffer_rsrc_t r0 = tile_rsrc(X, t0, n, ld);
        const __amdgpu_buffer_rsrc_t r1 = tile_rsrc(X, t0 + P, n, ld);
#pragma unroll
        for (int q = 0; q < K; ++q) preA[q] = load_quad(r0, xoff + 16 * q);
#pragma unroll
        for (int q = K; q < NQ; ++q) xv[q - K] = load_quad(r0, xoff + 16 * q);
#pragma unroll
        for (int q = 0; q < K; ++q) preB[q] = load_quad(r1, xoff + 16 * q);
        __syncthreads();  // LDS set up by the walkers
        if (sDone != 0) return;
        const char* cbase = reinterpret_cast<const char*>(sC + (lane < CPC ? lane : CPC - 1) * XS);
        float* myrow = tile + lane * XS;
        int changed = 0;

        auto round = [&](int r, float4* pre) {
            const long t = t0 + (long)r * P;
            const long nrow = n - t * 64 < 64 ? n - t * 64 : 64;
            const bool valid = lane < nrow;
            // the tile's labels; lanes past the last row fall outside the
            // descriptor (the load returns 0, the store is dropped)
            const __amdgpu_buffer_rsrc_t rl =
                __builtin_amdgcn_make_buffer_rsrc(labels + t * 64, (short)0, (int)(nrow * 4), 0x00020000);
            const int old = __builtin_amdgcn_raw_buffer_load_b32(rl, lane * 4, 0, 0);
            const __amdgpu_buffer_rsrc_t rn = tile_rsrc(X, t + P, n, ld);
            v4f acc[KG];
#pragma unroll
            for (int g = 0; g < KG; ++g) acc[g] = v4f{0.f, 0.f, 0.f, 0.f};
            float4 cv = *reinterpret_cast<const float4*>(cbase);
            int seen = 0;  // walker progress last read
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                // chunk q of the LDS tile is rewritten below once the walker
                // has read it for tile t - P (it runs well ahead: few polls)
                if (q >= K && r > 0) {
                    const int need = (r - 1) * NQ + q + 1;
                    if (seen < need) seen = wait_flag(&sProg[pair], need);
                }
                const float4 cvn = *reinterpret_cast<const float4*>(cbase + 16 * (q + 1 < NQ ? q + 1 : 0));
                const float4 x = q < K ? pre[q < K ? q : 0] : xv[q < K ? 0 : q - K];
                mfma_groups<KG>(acc, cv.x, x.x);
                mfma_groups<KG>(acc, cv.y, x.y);
                mfma_groups<KG>(acc, cv.z, x.z);
                mfma_groups<KG>(acc, cv.w, x.w);
                if (q >= K) {
                    *reinterpret_cast<float4*>(myrow + 4 * q) = x;
                    // tile t + P into the registers of the last LB chunks,
                    // back to back: the loads of one row's 16-byte pieces
                    // then meet the same cache lines together
                    if ((q - K) % LB == LB - 1 || q == NQ - 1) {
#pragma unroll
                        for (int qq = q - (q - K) % LB; qq <= q; ++qq) xv[qq - K] = load_quad(rn, xoff + 16 * qq);
                    }
                }
                cv = cvn;
                // one chunk per scheduling region: keeps each chunk's load
                // in its chunk, spreading the HBM reads over the E-step
                __builtin_amdgcn_sched_barrier(0);
            }
            // ||c||^2 - 2 x.c, first minimum wins (_k_means_lloyd.pyx:196-212)
            float d[CPC];
#pragma unroll
            for (int g = 0; g < KG; ++g) {
#pragma unroll
                for (int i = 0; i < 4; ++i) d[4 * g + i] = fmaf(-2.0f, acc[g][i], sN[4 * g + i]);
            }
            const int bidx = argmin_tree<CPC>(d);
            __builtin_amdgcn_raw_buffer_store_b32(bidx, rl, lane * 4, 0, 0);
            changed += (int)__popcll(__ballot(valid && old != bidx));
            // held chunks to LDS, then their registers take tile t + 2P
            const __amdgpu_buffer_rsrc_t rn2 = tile_rsrc(X, t + 2 * P, n, ld);
#pragma unroll
            for (int q = 0; q < K; ++q) {
                *reinterpret_cast<float4*>(myrow + 4 * q) = pre[q];
                pre[q] = load_quad(rn2, xoff + 16 * q);
            }
            // the tile's rows of each cluster
            if (lane < CPC) sMask[pair][lane] = 0ull;
            if (valid) atomicOr(&sMask[pair][bidx], 1ull << lane);
            set_flag(&sReady[pair], r + 1);
        };

        int r = 0;
        for (; r + 1 < rounds; r += 2) {
            round(r, preA);
            round(r + 1, preB);
        }
        if (r < rounds) round(r, preA);
        // one global atomic per block (below), not one per wave
        if (lane == 0 && changed != 0) atomicAdd(&sChg, changed);
        __syncthreads();  // every pair's walker is done: the tile area is free
        __syncthreads();  // the walkers' sums are in LDS
    } else {
        // walker waves: the halt test, then centres and the zero row into
        // LDS (all loads in flight at once) and ||c||^2
        const int prev = st->done;  // an earlier step halted the loop
        if (prev != 0) {
            if (tid == 256) sDone = prev;
            __syncthreads();
            return;
        }
        const int wt = tid - 256;
        constexpr int NF = (CPC * NQ + 255) / 256;
        float4 cf[NF];
#pragma unroll
        for (int u = 0; u < NF; ++u) {
            const int idx = wt + 256 * u;
            const int cl = idx / NQ;
            const int q = idx - cl * NQ;
            cf[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (idx < CPC * NQ && cl < k) cf[u] = *reinterpret_cast<const float4*>(C + (long)cl * ld + 4 * q);
        }
#pragma unroll
        for (int u = 0; u < NF; ++u) {
            const int idx = wt + 256 * u;
            const int cl = idx / NQ;
            const int q = idx - cl * NQ;
            if (idx < CPC * NQ) *reinterpret_cast<float4*>(&sC[cl * XS + 4 * q]) = cf[u];
        }
        for (int i = wt; i < XS; i += 256) zrow[i] = 0.f;
        if (wt < 4) {
            sReady[wt] = 0;
            sProg[wt] = 0;
        }
        if (wt == 0) sChg = 0;
        if (wave == 4) step_norms<CPC>(a, lane, sN, &sDone);
        __syncthreads();
        if (sDone != 0) return;
        // walker
        float4 S[NQ];
        int cnt;
        walk_tiles<CPC, WS, NQ, XS>(S, cnt, rounds, lane, &sReady[pair], &sProg[pair], sMask[pair], lbase, toff,
                                    zoff);
        __syncthreads();  // every pair is done with its tile
        publish_sums<CPC, NQ>(S, cnt, zrow + XS, ld, pair, lane, sCnt);
        __syncthreads();
    }
    if (tid == 0 && sChg != 0) atomicAdd(a.changed, sChg);
    combine_sums<CPC>(zrow + XS, ld, k, psum, pcnt, sCnt, tid, &st->present[a.iter & 1]);
}

// ---------------------------------------------------------------------------
// k_fused_low: rows of at most 16 floats
// ---------------------------------------------------------------------------
//
// Short rows leave little arithmetic per row, and k_fused's round (load, E-step,
// argmin, hand-over to the walker) is latency with two waves a SIMD: 33 us at
// 1M x 3, k = 64 and 71 us at 1M x 16, k = 20, for 16 and 64 MB.  Here every
// wave works alone, four a SIMD, with no hand-over: 64 R rows at a time, R
// rows a lane, the next ones in flight.  The E-step runs on the VALU (x.c as
// the fma chain over the features that the fp32 MFMAs make, then ||c||^2 - 2
// x.c and a strict '<' scan), the centres read from LDS as broadcasts, once
// per R rows (at R = 1 those reads take as long as the arithmetic).  The sums:
// per 64 rows an LDS bit mask of each cluster's rows; lane (cluster c, slice
// s) of 64 / KP slices (KP = k rounded up to a power of two) walks the slice's
// rows of c in ascending order.  Slices meet by an xor butterfly, waves in
// order: bitwise reproducible.  Bound by the VALU (k = 64) or HBM (k <= 8).
// LDS: centres [64][4 NQ] | per wave: rows [65][4 NQ] (the last one zeros), masks [64]
template <int NQ>
constexpr size_t low_wave_bytes()
{
    return 65 * 16 * NQ + 64 * sizeof(unsigned long long);
}

template <int NQ, int R>
__global__ __launch_bounds__(1024) void k_fused_low(FusedArgs a)
{
    constexpr int LD = 4 * NQ;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    __shared__ __attribute__((aligned(16))) float sN[64];
    __shared__ int sCnt[16][64];
    __shared__ int sDone, sChg;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = (int)(blockDim.x >> 6);
    const int k = a.k;
    const long n = a.n;
    float* const sC = lds;
    char* const mine = reinterpret_cast<char*>(lds + 64 * LD) + wave * low_wave_bytes<NQ>();
    f4v* const tile = reinterpret_cast<f4v*>(mine);
    unsigned long long* const mask = reinterpret_cast<unsigned long long*>(mine + 65 * 16 * NQ);
    // this wave's chunks of 64 R rows: c0, c0 + cstep, ..
    const long cstep = (long)gridDim.x * nw * (64 * R);
    long c0 = ((long)blockIdx.x * nw + wave) * (64 * R);
    f4v x[R][NQ], xn[R][NQ];
    int old[R], oldn[R];
    auto load = [&](long c) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const long row = min(c + 64 * r + lane, n - 1);
            const f4v* p = reinterpret_cast<const f4v*>(a.X + row * LD);
#pragma unroll
            for (int q = 0; q < NQ; ++q) xn[r][q] = p[q];
            oldn[r] = a.labels[row];
        }
    };
    if (c0 < n) load(c0);
    // centres (zeros past k: their norms are +inf), the zero row, norms and
    // the previous step's decision
    for (int i = tid; i < 64 * NQ; i += (int)blockDim.x) {
        const int j = i / NQ;
        f4v v = {0.f, 0.f, 0.f, 0.f};
        if (j < k) v = *reinterpret_cast<const f4v*>(a.C + (long)i * 4);
        *reinterpret_cast<f4v*>(sC + 4 * i) = v;
    }
    if (lane < NQ) tile[64 * NQ + lane] = f4v{0.f, 0.f, 0.f, 0.f};
    if (wave == 0) {
        const int prev = a.state->done;  // an earlier step halted the loop
        if (prev != 0) {
            if (lane == 0) sDone = prev;
        } else {
            step_norms<64>(a, lane, sN, &sDone);
        }
        if (lane == 0) sChg = 0;
    }
    __syncthreads();
    if (sDone != 0) return;
    int lk = 0;
    while ((1 << lk) < k) ++lk;
    const int KP = 1 << lk;
    const int c = lane & (KP - 1), sl = lane >> lk;
    const unsigned long long smask = KP == 64 ? ~0ull : (1ull << KP) - 1ull;  // a slice is KP rows
    f4v S[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) S[q] = f4v{0.f, 0.f, 0.f, 0.f};
    int cnt = 0, changed = 0;
    const int k4 = (k + 3) & ~3;
    for (; c0 < n; c0 += cstep) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) x[r][q] = xn[r][q];
            old[r] = oldn[r];
        }
        if (c0 + cstep < n) load(c0 + cstep);  // in flight while this chunk is worked on
        float best[R];
        int bi[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            best[r] = INFINITY;
            bi[r] = 0;
        }
        for (int j = 0; j < k4; j += 4) {
            const f4v cn = *reinterpret_cast<const f4v*>(sN + j);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                f4v cv[NQ];
#pragma unroll
                for (int q = 0; q < NQ; ++q) cv[q] = *reinterpret_cast<const f4v*>(sC + (j + u) * LD + 4 * q);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    float acc = 0.f;
#pragma unroll
                    for (int q = 0; q < NQ; ++q) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc = fmaf(x[r][q][e], cv[q][e], acc);
                    }
                    const float d = fmaf(-2.0f, acc, cn[u]);  // NaN compares false
                    const bool take = d < best[r];
                    best[r] = take ? d : best[r];
                    bi[r] = take ? j + u : bi[r];
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const long row = c0 + 64 * r + lane;
            const bool valid = row < n;
            if (valid) a.labels[row] = bi[r];
            changed += (int)__popcll(__ballot(valid && old[r] != bi[r]));
            // the 64 rows to LDS and the masks of each cluster's rows (a
            // wave's LDS accesses are performed in order)
#pragma unroll
            for (int q = 0; q < NQ; ++q) tile[lane * NQ + q] = x[r][q];
            if (lane < KP) mask[lane] = 0ull;
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_wave_barrier();
            if (valid) atomicOr(&mask[bi[r]], 1ull << lane);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_wave_barrier();
            const int r0 = sl << lk;
            unsigned long long m = (mask[c] >> r0) & smask;
            cnt += (int)__popcll(m);
            while (__ballot(m != 0ull) != 0ull) {
                // two rows at a time; past the last one the row of zeros
                int rr[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    rr[u] = m != 0ull ? r0 + __ffsll((long long)m) - 1 : 64;
                    m &= m - 1ull;
                }
                f4v v[2][NQ];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
#pragma unroll
                    for (int q = 0; q < NQ; ++q) v[u][q] = tile[rr[u] * NQ + q];
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
#pragma unroll
                    for (int q = 0; q < NQ; ++q) S[q] += v[u][q];
                }
            }
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_wave_barrier();
        }
    }
    // the slices of a cluster, then the waves in order
    for (int off = KP; off < 64; off <<= 1) {
        cnt += __shfl_xor(cnt, off, 64);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
#pragma unroll
            for (int e = 0; e < 4; ++e) S[q][e] += __shfl_xor(S[q][e], off, 64);
        }
    }
    if (lane == 0 && changed != 0) atomicAdd(&sChg, changed);
    __syncthreads();  // every wave is done with its rows
    float* const red = lds + 64 * LD;  // [wave][KP][LD]
    if (lane < KP) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) *reinterpret_cast<f4v*>(red + (wave * KP + lane) * LD + 4 * q) = S[q];
        sCnt[wave][lane] = cnt;
    }
    __syncthreads();
    if (tid == 0 && sChg != 0) atomicAdd(a.changed, sChg);
    float* const out = a.psum + (long)blockIdx.x * k * LD;
    for (int i = tid; i < k * LD; i += (int)blockDim.x) {
        float t = red[i];
        for (int w = 1; w < nw; ++w) t += red[w * KP * LD + i];
        out[i] = t;
    }
    if (tid < 64) {
        int t = 0;
        if (tid < k) {
            for (int w = 0; w < nw; ++w) t += sCnt[w][tid];
            a.pcnt[(long)blockIdx.x * k + tid] = t;
        }
        const unsigned long long m = __ballot(t > 0);
        if (tid == 0 && m != 0ull) atomicOr(&a.state->present[a.iter & 1], m);
    }
}

typedef void (*fused_fn)(FusedArgs);

// Whether k_fused_low takes the shape.  Its E-step is k (ld + 3) VALU
// instructions a row and wave, where k_fused's MFMA wave has the VALU to its
// argmin: few centres or features, and, while the walkers' rounds are what
// k_fused waits for, more rows.  Kernel times, k_fused / k_fused_low: 1M x 3:
// k = 64 33 / 24 us, k = 16 43 / 15, k = 4 28 / 13; 1M x 8: k = 64 39 / 32,
// k = 20 62 / 20; 1M x 16: k = 64 51 / 52, k = 20 71 / 31, k = 8 39 / 27;
// 50,000 rows: 3 floats, k = 64 8.1 / 9.7, k = 16 8.8 / 7.8; 8 floats, k = 64
// 8.3 / 10.7, k = 20 10.0 / 8.6; 16 floats, k = 64 9.6 / 13.0, k = 20 10.6 /
// 9.7.
static bool low_takes(long n, int ld, int k)
{
    const int ops = k * (ld + 3);
    return ld <= 16 && (ops <= 400 || (n >= 150000 && ops <= 750));
}

// Waves a block and rows a lane for n rows: four-wave blocks while every CU
// has at most one of them (the E-step's VALU time is per wave), else sixteen
// waves, and two rows a lane (which halve the LDS reads of the centres) once
// every wave has two tiles of 64.  Four rows a lane were no faster from 1M to
// 4M rows.
struct LowShape {
    int waves, rows;
};
static LowShape low_shape(long n, int num_cu)
{
    const long tiles = (n + 63) / 64;
    if (tiles <= 4L * num_cu) return {4, 1};
    return {16, tiles <= 32L * num_cu ? 1 : 2};
}

static fused_fn low_kernel(int ld, int rows)
{
    switch (ld) {
    case 4: return rows == 1 ? &k_fused_low<1, 1> : &k_fused_low<1, 2>;
    case 8: return rows == 1 ? &k_fused_low<2, 1> : &k_fused_low<2, 2>;
    case 16: return rows == 1 ? &k_fused_low<4, 1> : &k_fused_low<4, 2>;
    default: return nullptr;
    }
}

static size_t low_dyn_lds(int ld, int waves)
{
    const size_t per = ld == 4 ? low_wave_bytes<1>() : ld == 8 ? low_wave_bytes<2>() : low_wave_bytes<4>();
    return 64 * (size_t)ld * sizeof(float) + (size_t)waves * per;
}

template <int NQ, int... KGs>
struct FusedTable {
    static fused_fn get(int kg)
    {
        fused_fn f = nullptr;
        ((kg == KGs ? (f = &k_fused<KGs, NQ>, 0) : 0), ...);
        return f;
    }
};

template <int NQ>
static fused_fn pick_fused(int kg)
{
    return FusedTable<NQ, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16>::get(kg);
}

// Compiled row sizes (float4s); ld = 4 * NQ.
static fused_fn fused_kernel(int k, int ld)
{
    if (k < 1 || k > 64) return nullptr;
    const int kg = (k + 3) / 4;
    switch (ld) {
    case 4: return pick_fused<1>(kg);
    case 8: return pick_fused<2>(kg);
    case 16: return pick_fused<4>(kg);
    case 32: return pick_fused<8>(kg);
    case 48: return pick_fused<12>(kg);
    case 64: return pick_fused<16>(kg);
    case 80: return pick_fused<20>(kg);
    case 100: return pick_fused<25>(kg);
    default: return nullptr;
    }
}
static size_t fused_dyn_lds(int k, int ld)
{
    const int cpc = 4 * ((k + 3) / 4);
    return (size_t)(cpc + 1 + 4 * 64) * fused_stride(ld / 4) * sizeof(float);
}

int fused_ld(int d, int k)
{
    // SKMETAL_HIP_FUSED=0 selects the separate assign/update kernels for every shape
    const char* env = getenv("SKMETAL_HIP_FUSED");
    if (env != nullptr && env[0] == '0') return 0;
    if (d < 1 || k < 1 || k > 64) return 0;
    static const int kLds[] = {4, 8, 16, 32, 48, 64, 80, 100};
    for (int ld : kLds) {
        if (ld < d) continue;
        if (ld <= 16) {
            for (const int rows : {1, 2}) {
                if (hipFuncSetAttribute(reinterpret_cast<const void*>(low_kernel(ld, rows)),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)low_dyn_lds(ld, 16)) !=
                    hipSuccess) {
                    (void)hipGetLastError();
                    return 0;
                }
            }
        }
        fused_fn f = fused_kernel(k, ld);
        const size_t dyn = fused_dyn_lds(k, ld);
        const size_t stat = 4 * 64 * (sizeof(unsigned long long) + sizeof(int)) + 64 * sizeof(float);  // sMask, sCnt, sN
        if (f == nullptr || dyn + stat > 160 * 1024) return 0;
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(f), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)dyn) != hipSuccess) {
            (void)hipGetLastError();
            return 0;
        }
        return ld;
    }
    return 0;
}

int fused_blocks(long n, int ld, int k, int num_cu)
{
    const long tiles = (n + 63) / 64;
    if (low_takes(n, ld, k)) {
        const LowShape g = low_shape(n, num_cu);
        const long blocks = (tiles + g.waves * g.rows - 1) / (g.waves * g.rows);
        return (int)(blocks < 1 ? 1 : blocks < num_cu ? blocks : num_cu);
    }
    if (fused_kernel(k, ld) == nullptr) return 0;
    long blocks = (tiles + 3) / 4;
    if (blocks > num_cu) blocks = num_cu;
    return (int)(blocks < 1 ? 1 : blocks);
}

hipError_t launch_fused(const FusedArgs& a, hipStream_t s)
{
    if (a.split) return launch_fused3(a, s);
    if (low_takes(a.n, a.ld, a.k)) {
        if (a.blocks < 1 || a.k < 1 || a.k > 64) return hipErrorInvalidValue;
        const LowShape g = low_shape(a.n, a.num_cu);
        const fused_fn f = low_kernel(a.ld, g.rows);
        if (f == nullptr) return hipErrorInvalidValue;
        hipLaunchKernelGGL(f, dim3(a.blocks), dim3(64 * g.waves), low_dyn_lds(a.ld, g.waves), s, a);
        return hipGetLastError();
    }
    fused_fn f = fused_kernel(a.k, a.ld);
    if (f == nullptr || a.blocks < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(f, dim3(a.blocks), dim3(512), fused_dyn_lds(a.k, a.ld), s, a);
    return hipGetLastError();
}
}  // namespace skm
