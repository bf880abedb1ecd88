// drain_scan.hip -- whole-ring drain of SSLA-S s2 + s3 + YOLOX head on gfx950.
//
// The reference drains a ring 8 records at a time in one 9-warp block per
// ring (orin/kernels/ssla_s2_s3_head_celled.cuh:914-1255), so at most 8
// records are in flight per block.  This file re-derives the same result
// for a whole pre-filled ring at once, using the structure of one SSLA layer
// (orin/orin/ssla_ref.py:17-93):
//
//   for every in-bounds patch cell c of event e (offset delta):
//       q, v, g = qvgIn[delta] x_e                    (depends on x_e only)
//       h_c     = sigmoid(g) * h_c + v                (ordered per cell)
//       qh      = q * h_c
//   y_e = LN( sum_delta goW[delta] qh + residual(x_e) )
//
// Only the h_c recurrence is ordered, and only among events touching the
// same cell.  Per layer the drain therefore runs two kernels over all records
// of all rings:
//   P, S (k_pscan)  v, g for every (record, delta) pair as MFMA tiles, and the
//                   recurrence over them: groups of pairs in per-cell ring
//                   order, chained by a look-back scan; writes the h rows
//                   where the layer's output is used
//   O    (k_outt)   per output record: q = qvgIn[delta] x by MFMA, times the
//                   <= 9 h rows, contracted with goW by MFMA, residual, fp64
//                   LayerNorm
// The temporal-dropout decisions (ssla_ref.py:190-195) depend only on the
// per-cell arrival rank of a record, so they come from a stable sort of
// records by cell: pass = ((counter + rank) mod 256) % window == 0.
// Results equal sequential processing in ring order up to fp32 summation
// order; drop decisions are bit-exact.
//
// Device layouts are those of include/ssla_abi.h.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <atomic>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "drain_common.h"
#include "drain_scan.h"
#include "mfma_pack.h"

namespace ssla {

namespace {


struct BlockDesc {
    const HybridInputRec* ring;
    HybridS2S3OutputSlot* out;
    float*                head_out;
    float*                hidden[4];
    unsigned char*        td2;
    unsigned char*        td3;
    float*                preds;
    unsigned int*         version;
    HybridStrip           strip;
    int                   n;
    int                   offset;
};

// The block table travels to the device as kernel arguments of k_decode
// (the runtime copies them at launch, so a call never waits on the host for
// a staging buffer the previous call may still be reading); k_decode reads
// it there and writes the copy the later kernels read.
struct BlockTable {
    BlockDesc d[SSLA_MAX_BLOCKS];
};
static_assert(sizeof(BlockTable) <= 2048, "kernel argument block");

__device__ __forceinline__ int find_block(const BlockDesc* bd, int nb, int g) {
    int b = 0;
    for (int i = 1; i < nb; ++i)
        if (g >= bd[i].offset) b = i;
    return b;
}

// ---------------------------------------------------------------------------
// decode: ring records -> compact features, centre cells, sort keys
// ---------------------------------------------------------------------------
// Eight lanes per 128-byte record, one 16-byte load each: lanes 1..6 move the
// feat1 quarters, lane 0 also writes the keys.
constexpr int kDecRec = 32;          // records per 256-thread workgroup

// Up to kFills int arrays set to a value each (k_decode's extra blocks).
constexpr int kFills = 7;
struct FillSet {
    int* p[kFills];
    int n[kFills];
    int v[kFills];
};

// One launch for the call's set-up: blocks [0, ndec) decode the records,
// then fblk blocks per fill array, then npk blocks rebuild the fragment-order
// weight copies (one float per thread), and the last block writes the block
// table for the later kernels.  Nothing in this launch reads what another of
// its blocks writes.
__global__ void __launch_bounds__(256)
k_decode(int E, BlockTable tab, BlockDesc* __restrict__ bd_out, Geometry G,
         float* __restrict__ X0, int* __restrict__ cell2,
         unsigned char* __restrict__ owner,
         uint32_t* __restrict__ key2, uint32_t* __restrict__ val2, int ndec, FillSet f, int fblk,
         PackSrc ps, float* __restrict__ pbuf, int npk) {
    const int nfill = fblk * kFills;
    if ((int)blockIdx.x >= ndec) {
        const int xb = (int)blockIdx.x - ndec;
        if (xb < nfill) {
            // the call's fills: fblk blocks of 256 per array
            const int a = xb / fblk;
            const int i = (xb - a * fblk) * 256 + (int)threadIdx.x;
            if (i < f.n[a]) f.p[a][i] = f.v[a];
        } else if (xb < nfill + npk) {
            const size_t q = (size_t)(xb - nfill) * 256 + threadIdx.x;
            if (q < PackLayout<true>::off[8]) pack_elem<true>(ps, pbuf, q);
        } else if (threadIdx.x < SSLA_MAX_BLOCKS) {
            bd_out[threadIdx.x] = tab.d[threadIdx.x];
        }
        return;
    }
    const int g = blockIdx.x * kDecRec + (threadIdx.x >> 3);
    const int c = threadIdx.x & 7;
    if (g >= E) return;
    int b = 0;
    for (int i = 1; i < G.nb; ++i)
        if (g >= tab.d[i].offset) b = i;
    const HybridInputRec* r = tab.d[b].ring + (g - tab.d[b].offset);
    const float4 v = reinterpret_cast<const float4*>(r)[c];
    const int x = r->x, y = r->y;
    const bool valid = x < G.W2 && y < G.H2;
    if (c >= 1 && c <= SSLA_C1 / 4)
        reinterpret_cast<float4*>(X0 + (size_t)g * SSLA_C1)[c - 1] =
            valid ? v : make_float4(0.f, 0.f, 0.f, 0.f);
    if (c != 0) return;
    const HybridStrip& s = tab.d[b].strip;
    owner[g] = (valid && x >= s.owned_lo && x < s.owned_hi &&
                y >= s.owned_y_lo && y < s.owned_y_hi) ? 1 : 0;
    const uint32_t none = (uint32_t)(G.nb * G.C2);
    cell2[g] = valid ? y * G.W2 + x : -1;
    key2[g] = valid ? (uint32_t)(b * G.C2 + y * G.W2 + x) : none;
    val2[g] = (uint32_t)g;
}



// ---------------------------------------------------------------------------
// Stable LSD radix sort of (key, record) pairs, digits of up to 9 bits.
// Records are taken in tiles of kRTile (256 threads x 8 rounds, round r =
// records base + 256 r .. + 255).  Per pass:
//   k_rs_hist     digit counts of every tile            -> bh[digit * T + tile]
//   k_exscan      exclusive scan of bh (digit-major)    -> first slot of every
//                                                          (digit, tile)
//   k_rs_scatter  each record to its (digit, tile) start + its rank among
//                 the tile's earlier records of the digit: inside a wave from
//                 the lanes whose digit equals its own (one ballot per digit
//                 bit), across the round's waves and rounds from LDS counts.
// ---------------------------------------------------------------------------
constexpr int kRThreads = 256, kRRounds = 8, kRTile = kRThreads * kRRounds;
constexpr int kRMaxBits = 9;

__global__ void __launch_bounds__(kRThreads)
k_rs_hist(int n, const uint32_t* __restrict__ keys, int shift, int bits, int nbins, int T,
          int* __restrict__ bh) {
    __shared__ int h[1 << kRMaxBits];
    const int nb = 1 << bits, tid = threadIdx.x;
    for (int i = tid; i < nb; i += kRThreads) h[i] = 0;
    __syncthreads();
    const int base = blockIdx.x * kRTile;
    #pragma unroll 4
    for (int r = 0; r < kRRounds; ++r) {
        const int idx = base + r * kRThreads + tid;
        if (idx < n) atomicAdd(&h[(keys[idx] >> shift) & (nb - 1)], 1);
    }
    __syncthreads();
    for (int i = tid; i < nbins; i += kRThreads) bh[(size_t)i * T + blockIdx.x] = h[i];
}

// vin null: the values are the record indices.  sidx (last pass, optional):
// sidx[value] = the value's sorted position.
__global__ void __launch_bounds__(kRThreads)
k_rs_scatter(int n, const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
             uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, int* __restrict__ sidx,
             int shift, int bits, int nbins, int T, const int* __restrict__ boff) {
    __shared__ int cnt[1 << kRMaxBits];
    __shared__ int wcnt[kRThreads / 64][1 << kRMaxBits];
    const int nb = 1 << bits, tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    for (int i = tid; i < nbins; i += kRThreads) {
        cnt[i] = boff[(size_t)i * T + blockIdx.x];
        #pragma unroll
        for (int w = 0; w < kRThreads / 64; ++w) wcnt[w][i] = 0;
    }
    __syncthreads();
    const unsigned long long below = (1ull << lane) - 1ull;
    const int base = blockIdx.x * kRTile;
    for (int r = 0; r < kRRounds; ++r) {
        const int idx = base + r * kRThreads + tid;
        const bool valid = idx < n;
        const uint32_t key = valid ? kin[idx] : 0u;
        const int dig = (int)((key >> shift) & (uint32_t)(nb - 1));
        unsigned long long peers = __ballot(valid);
        for (int b = 0; b < bits; ++b) {
            const bool bit = (dig >> b) & 1;
            const unsigned long long m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const int rank = __popcll(peers & below), size = __popcll(peers);
        const bool leader = valid && rank == 0;
        if (leader) wcnt[wv][dig] = size;
        __syncthreads();
        if (valid) {
            int pos = cnt[dig] + rank;
            for (int w = 0; w < wv; ++w) pos += wcnt[w][dig];
            const uint32_t v = vin ? vin[idx] : (uint32_t)idx;
            kout[pos] = key;
            vout[pos] = v;
            if (sidx) sidx[v] = pos;
        }
        __syncthreads();
        if (leader) {
            atomicAdd(&cnt[dig], size);
            wcnt[wv][dig] = 0;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// One workgroup scans arrays of any length in rounds of kScanThreads x 8
// elements: each thread loads 8 consecutive elements with two 16-byte loads,
// the thread totals are scanned in LDS, and a running carry joins the rounds.
// Arrays are 256-byte aligned workspace buffers (16-byte loads stay in them;
// elements at or past n read as zero and are not written).
// ---------------------------------------------------------------------------
constexpr int kScanThreads = 1024, kScanPer = 8, kScanRound = kScanThreads * kScanPer;

// exclusive prefix of v over the workgroup; *total receives the sum
__device__ __forceinline__ int block_exscan(int v, int* lds, int* total) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    int x = v;
    #pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) lds[wv] = x;
    __syncthreads();
    if (wv == 0) {
        int w = lane < kScanThreads / 64 ? lds[lane] : 0;
        #pragma unroll
        for (int o = 1; o < kScanThreads / 64; o <<= 1) {
            const int y = __shfl_up(w, o, 64);
            if (lane >= o) w += y;
        }
        if (lane < kScanThreads / 64) lds[kScanThreads / 64 + lane] = w;
    }
    __syncthreads();
    const int before = (wv ? lds[kScanThreads / 64 + wv - 1] : 0) + x - v;
    *total = lds[2 * (kScanThreads / 64) - 1];
    __syncthreads();
    return before;
}

__device__ __forceinline__ void load8(const int* a, int i0, int n, int (&v)[kScanPer]) {
    if (i0 + kScanPer <= n) {
        const int4 x = reinterpret_cast<const int4*>(a + i0)[0];
        const int4 y = reinterpret_cast<const int4*>(a + i0)[1];
        v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
        v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
    } else {
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q) v[q] = i0 + q < n ? a[i0 + q] : 0;
    }
}

__device__ __forceinline__ void store8(int* a, int i0, int n, const int (&v)[kScanPer]) {
    if (i0 + kScanPer <= n) {
        reinterpret_cast<int4*>(a + i0)[0] = make_int4(v[0], v[1], v[2], v[3]);
        reinterpret_cast<int4*>(a + i0)[1] = make_int4(v[4], v[5], v[6], v[7]);
    } else {
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q)
            if (i0 + q < n) a[i0 + q] = v[q];
    }
}

// in place: a[i] <- sum of a[0 .. i)
__global__ void __launch_bounds__(kScanThreads) k_exscan(int n, int* __restrict__ a) {
    __shared__ int lds[2 * (kScanThreads / 64)];
    int carry = 0;
    for (int r0 = 0; r0 < n; r0 += kScanRound) {
        const int i0 = r0 + (int)threadIdx.x * kScanPer;
        int v[kScanPer];
        load8(a, i0, n, v);
        int sum = 0;
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q) sum += v[q];
        int total;
        int run = carry + block_exscan(sum, lds, &total);
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q) {
            const int x = v[q];
            v[q] = run;
            run += x;
        }
        store8(a, i0, n, v);
        carry += total;
    }
}

// Groups of the projection + scan kernel (k_pscan): a cell with more than
// kGW pairs is cut into groups of kGP of its own; cells with fewer share one,
// all those whose run starts in the same window of kGW pair positions (runs
// of the pair order are contiguous, and a cell that starts in a window behind
// a larger one starts in a later window, so a shared group is one range of at
// most 2 kGW - 1 pairs).
constexpr int kGP = 176;        // pairs per group (k_pscan: 4 row blocks of 44 per channel)
constexpr int kGW = kGP / 2;

// group list entry: {first pair, pairs | flags, published-word slot, rank in the cell}
constexpr int kGStart = 1 << 16;    // the group's first pair is its cell's first
constexpr int kGEnd = 1 << 17;      // the group's last pair is its cell's last
constexpr int kGMulti = 1 << 18;    // the group holds several cells

// first index in [lo, hi) of the ascending array a whose value is >= v, else hi
__device__ __forceinline__ int lower_bound_i(const int* a, int lo, int hi, int v) {
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// The groups that key k leads (pst: nk + 1 pair starts): its count, and the
// end of their pair range.
__device__ __forceinline__ int key_groups(int k, int nk, const int* pst, int* pend) {
    const int s = pst[k], e = pst[k + 1], n = e - s;
    *pend = e;
    if (n == 0) return 0;
    if (n > kGW) return (n + kGP - 1) / kGP;
    const int w0 = s - s % kGW;
    if (pst[lower_bound_i(pst, 0, k, w0)] != s) return 0;     // an earlier cell of the window leads
    const int kb = lower_bound_i(pst, k + 1, nk, min(w0 + kGW, pst[nk]));
    // key kb - 1 is the last with pairs that starts in the window
    *pend = pst[kb] - pst[kb - 1] > kGW ? pst[kb - 1] : pst[kb];
    return 1;
}

// Per key, for the keys k_keyscan has no room for in LDS: the groups it leads
// (gcnt), the end of their range (gend) and its place among the keys with as
// many (ghist counts them).
__device__ __forceinline__ void key_group_at(uint32_t k, uint32_t nk, const int* __restrict__ pst,
                                             int* __restrict__ gcnt, int* __restrict__ gend,
                                             int* __restrict__ ghist, int* __restrict__ gw) {
    if (k >= nk) return;
    int pend;
    const int gc = key_groups((int)k, (int)nk, pst, &pend);
    gcnt[k] = gc;
    gend[k] = pend;
    if (gc > 0) gw[k] = atomicAdd(&ghist[gc], 1);
}

__global__ void __launch_bounds__(256)
k_key_groups(uint32_t nk, const int* __restrict__ pst, int* __restrict__ gcnt,
             int* __restrict__ gend, int* __restrict__ ghist, int* __restrict__ gw) {
    key_group_at(blockIdx.x * 256u + threadIdx.x, nk, pst, gcnt, gend, ghist, gw);
}

// The ticket order of the groups (one workgroup): tickets take every cell's
// group 0, then every cell's group 1, ..., cells with more groups first, so
// a group's predecessors in its cell hold smaller tickets.  hist[v] counts the
// keys that lead v groups (nv entries) and place(k) is key k's place among
// them.  start[v] = keys with more than v groups (the groups of rank v),
// base[r] = tickets before rank r; key k, at place start[gc] + place of every
// rank below gc, gets glist[base[r] + start[gc] + place] for its rank r.
// lead(k) -> (group count, range end, place, first pair, first slot).
struct LeadKey {
    int gc, pend, place, p0, slot, multi;
};
template <class Lead>
__device__ __forceinline__ void group_order(int nk, int nv, const int* hist, int* start, int* base,
                                            int* lds, Lead lead, int4* __restrict__ glist,
                                            int* __restrict__ n_groups) {
    int carry = 0;
    for (int r0 = 0; r0 < nv; r0 += kScanRound) {        // start: scan of hist from the top
        const int i0 = r0 + (int)threadIdx.x * kScanPer;
        int v[kScanPer], sum = 0;
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q) {
            v[q] = i0 + q < nv ? hist[nv - 1 - (i0 + q)] : 0;
            sum += v[q];
        }
        int total;
        int run = carry + block_exscan(sum, lds, &total);
        carry += total;
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q) {
            if (i0 + q < nv) start[nv - 1 - (i0 + q)] = run;
            run += v[q];
        }
    }
    __syncthreads();
    carry = 0;
    for (int r0 = 0; r0 < nv; r0 += kScanRound) {        // base: prefix of start
        const int i0 = r0 + (int)threadIdx.x * kScanPer;
        int v[kScanPer], sum = 0;
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q) {
            v[q] = i0 + q < nv ? start[i0 + q] : 0;
            sum += v[q];
        }
        int total;
        int run = carry + block_exscan(sum, lds, &total);
        carry += total;
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q) {
            if (i0 + q < nv) base[i0 + q] = run;
            run += v[q];
        }
    }
    if (threadIdx.x == 0) *n_groups = carry;
    __syncthreads();
    for (int k = threadIdx.x; k < nk; k += kScanThreads) {
        const LeadKey L = lead(k);
        const int p = L.gc > 0 ? start[L.gc] + L.place : 0;
        for (int r = 0; r < L.gc; ++r) {
            const int p0 = L.p0 + r * kGP;
            glist[base[r] + p] = make_int4(p0, min(kGP, L.pend - p0) | (r == 0 ? kGStart : 0) |
                                                   (r == L.gc - 1 ? kGEnd : 0) | L.multi,
                                           L.slot + r, r);
        }
    }
}

// The same from the tables in global memory (any number of keys and groups).
__global__ void __launch_bounds__(kScanThreads)
k_group_order(int nk, int nv, const int* __restrict__ pst, const int* __restrict__ goff,
              const int* __restrict__ gcnt, const int* __restrict__ gend, const int* ghist,
              const int* __restrict__ gw, int* gstart, int* gbase, int4* __restrict__ glist,
              int* __restrict__ n_groups) {
    __shared__ int lds[2 * (kScanThreads / 64)];
    group_order(nk, nv, ghist, gstart, gbase, lds, [&](int k) {
        return LeadKey{gcnt[k], gend[k], gw[k], pst[k], goff[k],
                       gend[k] > pst[k + 1] ? kGMulti : 0};
    }, glist, n_groups);
}

// [start, end) of every key present in a sorted key array.
__global__ void k_runs(int n, const uint32_t* __restrict__ keys, uint32_t nk,
                       int* __restrict__ start, int* __restrict__ end) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t k = keys[p];
    if (k >= nk) return;
    if (p == 0 || keys[p - 1] != k) start[k] = p;
    if (p == n - 1 || keys[p + 1] != k) end[k] = p + 1;
}

// ---------------------------------------------------------------------------
// Temporal dropout (ssla_ref.py:190-195): a cell's counter c (uint8) takes
// pre = c + rank (mod 256) for the record of arrival rank `rank`, and the
// record passes when window <= 1 or pre % window == 0.  passes(c, r, w) is
// the number of passing ranks in [0, r): with F(x) = the number of
// u in [0, x) whose (u mod 256) is a multiple of w,
//   F(x) = (x / 256) (255 / w + 1) + ceil((x mod 256) / w),
// passes(c, r, w) = F(c + r) - F(c).
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool tdrop_pass(unsigned c, unsigned rank, int window) {
    return window <= 1 || ((c + rank) & 255u) % (unsigned)window == 0u;
}

__device__ __forceinline__ int tdrop_passes(unsigned c, int r, int window) {
    if (window <= 1) return r;
    const unsigned w = (unsigned)window, per = 255u / w + 1u;
    auto F = [&](unsigned x) { return (x >> 8) * per + ((x & 255u) + w - 1u) / w; };
    return (int)(F(c + (unsigned)r) - F(c));
}

// tdrop_s2 over the sorted records (position p, record g, rank r in the
// key's run, counter c before the call): pass2[g], and the pass-2 list in
// s2 order -- the record's place is the key's offset plus the number of
// passing ranks below r.  Returns pass2[g].
__device__ __forceinline__ bool
tdrop2_at(int p, int n, const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
          uint32_t nk, const int* __restrict__ start, const unsigned char* __restrict__ old,
          const int* __restrict__ off, int window, unsigned char* __restrict__ pass,
          int* __restrict__ list) {
    if (p >= n) return false;
    const uint32_t k = keys[p];
    const int g = (int)vals[p];
    if (k >= nk) {
        pass[g] = 0;
        return false;
    }
    const int r = p - start[k];
    const unsigned c = old[k];
    const bool take = tdrop_pass(c, (unsigned)r, window);
    pass[g] = take ? 1 : 0;
    if (take) list[off[k] + tdrop_passes(c, r, window)] = g;
    return take;
}


// Per s2 key: the counter before this call (old[k]), the counter after it,
// the number of pass-2 records of the run (n2[k]) and the pair count of the
// key (the run lengths of its 3 x 3 neighbourhood).
__global__ void k_keys2(uint32_t nk, int C, int W, int H, const int* __restrict__ st,
                        const int* __restrict__ en, const BlockDesc* __restrict__ bd, int window,
                        unsigned char* __restrict__ old, int* __restrict__ n2,
                        int* __restrict__ pcnt) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nk) return;
    const int b = (int)t / C, cell = (int)t % C, ty = cell / W, tx = cell % W;
    const int len = en[t] - st[t];
    unsigned char* td = bd[b].td2 + cell;
    const unsigned c = *td;
    old[t] = (unsigned char)c;
    n2[t] = tdrop_passes(c, len, window);
    *td = (unsigned char)((c + (unsigned)len) & 255u);
    int np = 0;
    #pragma unroll
    for (int oy = -1; oy <= 1; ++oy)
        #pragma unroll
        for (int ox = -1; ox <= 1; ++ox) {
            const int sy = ty + oy, sx = tx + ox;
            if (sy < 0 || sy >= H || sx < 0 || sx >= W) continue;
            const int s = b * C + sy * W + sx;
            np += en[s] - st[s];
        }
    pcnt[t] = np;
}

// The per-key tables of k_keys2 (and k_runs) for a one-pass record sort,
// whose digit is the whole key: the scanned tile histogram bh (bin-major, T
// tiles) holds the run bounds, key t's run being [bh[t T], bh[(t + 1) T]).
// key2_at writes st / en / old and the committed counter, and returns the
// key's pair count and pass-2 count (used by k_keyscan<true>).
struct KeyHist {
    int C, W, H, T, window;
    const int* bh;
    int* st;
    int* en;
    const BlockDesc* bd;
    unsigned char* old;
};

__device__ __forceinline__ void key2_at(uint32_t t, const KeyHist& kh, int& pc, int& n2v) {
    const int b = (int)t / kh.C, cell = (int)t % kh.C, ty = cell / kh.W, tx = cell % kh.W;
    const int s0 = kh.bh[(size_t)t * kh.T], len = kh.bh[(size_t)(t + 1) * kh.T] - s0;
    kh.st[t] = s0;
    kh.en[t] = s0 + len;
    unsigned char* td = kh.bd[b].td2 + cell;
    const unsigned c = *td;
    kh.old[t] = (unsigned char)c;
    n2v = tdrop_passes(c, len, kh.window);
    *td = (unsigned char)((c + (unsigned)len) & 255u);
    int np = 0;
    #pragma unroll
    for (int oy = -1; oy <= 1; ++oy)
        #pragma unroll
        for (int ox = -1; ox <= 1; ++ox) {
            const int sy = ty + oy, sx = tx + ox;
            if (sy < 0 || sy >= kh.H || sx < 0 || sx >= kh.W) continue;
            const size_t q = (size_t)(b * kh.C + sy * kh.W + sx);
            np += kh.bh[(q + 1) * kh.T] - kh.bh[q * kh.T];
        }
    pc = np;
}

// Per-key tables from per-key counts (k < nk), in one launch:
//   cnt  -> start (exclusive scan, nk + 1 values), end = start + cnt (optional;
//           end may be cnt itself);
//           with goff: goff[k] = the key's first published-word slot (one per
//           kGP pairs);
//   cnt2 (optional) -> off2 (exclusive scan), *total2.
// KH: the counts come from key2_at (a one-pass sort's histogram, kh; nk <=
// kScanThreads) instead of cnt / cnt2, and cnt2 then receives the pass-2
// counts.
// GT: the group list too (nk <= kScanThreads keys and gt.nv <= kGroupLds group
// counts, all tables in LDS), which a call with few keys would otherwise wait
// for two more launches for.
constexpr int kGroupLds = 6144;
struct GroupTab {
    int nv;
    int4* glist;
    int* n_groups;
};

// The group list of at most kScanThreads keys (one per thread of the
// workgroup) from pair starts pst (nk + 1) and word slots go; hist and start
// hold gt.nv entries, hist zero before.  All arrays in LDS.
__device__ __forceinline__ void group_list_lds(int nk, const int* pst, const int* go, int* hist,
                                               int* start, int* lds, GroupTab gt) {
    const int k = (int)threadIdx.x;
    int gc = 0, pend = 0, place = 0;
    if (k < nk) gc = key_groups(k, nk, pst, &pend);
    if (gc > 0) place = atomicAdd(&hist[gc], 1);
    __syncthreads();
    // (the base table takes hist's place: hist is read before it is written)
    group_order(nk, gt.nv, hist, start, hist, lds, [&](int q) {
        return LeadKey{gc, pend, place, pst[q], go[q], pend > pst[q + 1] ? kGMulti : 0};
    }, gt.glist, gt.n_groups);
}

template <bool KH, bool GT>
__global__ void __launch_bounds__(kScanThreads)
k_keyscan(int nk, const int* cnt, int* __restrict__ start, int* end, int* __restrict__ goff,
          const int* __restrict__ cnt2, int* __restrict__ off2,
          int* __restrict__ total2, KeyHist kh, GroupTab gt) {
    __shared__ int lds[2 * (kScanThreads / 64)];
    __shared__ int kv[KH ? kScanThreads : 1], ku[KH ? kScanThreads : 1];
    __shared__ int spst[GT ? kScanThreads + 1 : 1], sgo[GT ? kScanThreads : 1];
    __shared__ int shist[GT ? kGroupLds : 1], sstart[GT ? kGroupLds : 1];
    if constexpr (GT)
        for (int i = threadIdx.x; i < gt.nv; i += kScanThreads) shist[i] = 0;
    int carry = 0, ccarry = 0, carry2 = 0;
    for (int r0 = 0; r0 < nk; r0 += kScanRound) {
        const int i0 = r0 + (int)threadIdx.x * kScanPer;
        int v[kScanPer], c[kScanPer], u[kScanPer];
        if constexpr (KH) {
            // one key per thread (nk <= kScanThreads), through LDS into the
            // eight-per-thread layout of the scan
            const int t = (int)threadIdx.x;
            int pc = 0, p2 = 0;
            if (t < nk) {
                key2_at((uint32_t)t, kh, pc, p2);
                const_cast<int*>(cnt2)[t] = p2;
            }
            kv[t] = pc;
            ku[t] = p2;
            __syncthreads();
            #pragma unroll
            for (int q = 0; q < kScanPer; ++q) {
                const bool in = i0 + q < kScanThreads;
                v[q] = in ? kv[i0 + q] : 0;
                u[q] = in ? ku[i0 + q] : 0;
            }
        } else {
            load8(cnt, i0, nk, v);
            if (cnt2) load8(cnt2, i0, nk, u);
        }
        int s = 0, sc = 0, su = 0;
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q) {
            s += v[q];
            c[q] = (v[q] + kGP - 1) / kGP;
            sc += c[q];
            if (cnt2) su += u[q];
        }
        int total;
        int run = carry + block_exscan(s, lds, &total);
        carry += total;
        int crun = 0, urun = 0;
        if (goff) {
            crun = ccarry + block_exscan(sc, lds, &total);
            ccarry += total;
        }
        if (cnt2) {
            urun = carry2 + block_exscan(su, lds, &total);
            carry2 += total;
        }
        int st[kScanPer], en[kScanPer];
        #pragma unroll
        for (int q = 0; q < kScanPer; ++q) {
            st[q] = run;
            run += v[q];
            en[q] = run;
            const int x = c[q];
            c[q] = crun;
            crun += x;
            const int y = u[q];
            u[q] = urun;
            urun += y;
            if constexpr (GT) {
                if (i0 + q < nk) {
                    spst[i0 + q] = st[q];
                    sgo[i0 + q] = c[q];
                }
            }
        }
        store8(start, i0, nk, st);
        if (end) store8(end, i0, nk, en);
        if (goff) store8(goff, i0, nk, c);
        if (cnt2) store8(off2, i0, nk, u);
    }
    if (threadIdx.x == 0) {
        start[nk] = carry;
        if (cnt2) *total2 = carry2;
    }
    if constexpr (GT) {
        if (threadIdx.x == 0) spst[nk] = carry;
        __syncthreads();
        group_list_lds(nk, spst, sgo, shist, sstart, lds, gt);
    }
}

// Per s3 key: the number of pass-2 records of its four s2 cells (t3, the
// length of its run in the s3 order) and how many of them pass tdrop_s3.
__global__ void k_keys3a(uint32_t nk3, Geometry G, const int* __restrict__ n2,
                         const BlockDesc* __restrict__ bd, int* __restrict__ t3,
                         int* __restrict__ n3) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nk3) return;
    const int b = (int)k / G.C3, cell = (int)k % G.C3;
    const int x = 2 * (cell % G.W3), y = 2 * (cell / G.W3);
    const int s = b * G.C2 + y * G.W2 + x;
    const int t = n2[s] + n2[s + 1] + n2[s + G.W2] + n2[s + G.W2 + 1];
    t3[k] = t;
    n3[k] = tdrop_passes(bd[b].td3[cell], t, G.window);
}

// Lower bound of g in vals[lo, lo + len): the index of the first value >= g.
__device__ __forceinline__ int lower_bound_u32(const uint32_t* __restrict__ vals, int lo, int len,
                                               uint32_t g) {
    while (len > 0) {
        const int half = len >> 1;
        if (vals[lo + half] < g) {
            lo += half + 1;
            len -= half + 1;
        } else {
            len = half;
        }
    }
    return lo;
}

// The s3 order of the pass-2 records without a sort: a pass-2 record's rank
// in its s3 cell is the number of pass-2 records before it (record order)
// in the four s2 runs of that cell.  In its own run that is the number of
// passing ranks below its own; in the other three it is the number of
// passing ranks below its lower bound there.  Slot = start3 + rank:
// keys3 / vals3 is the s3 record order, key3g the record's s3 key.
__global__ void __launch_bounds__(256)
k_place3(const int* __restrict__ n_dev, const int* __restrict__ list,
         const BlockDesc* __restrict__ bd, Geometry G, const int* __restrict__ cell2,
         const int* __restrict__ sidx, const uint32_t* __restrict__ vals2,
         const int* __restrict__ st2, const int* __restrict__ en2,
         const unsigned char* __restrict__ old2, const int* __restrict__ st3,
         uint32_t* __restrict__ keys3, uint32_t* __restrict__ vals3,
         uint32_t* __restrict__ key3g) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= *n_dev) return;
    const int g = list[j];
    const int b = find_block(bd, G.nb, g);
    const int cell = cell2[g], x = cell % G.W2, y = cell / G.W2;
    const int k2 = b * G.C2 + cell;
    const int x0 = x & ~1, y0 = y & ~1;
    const uint32_t k3 = (uint32_t)(b * G.C3 + (y >> 1) * G.W3 + (x >> 1));
    int rank = 0;
    #pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int s = b * G.C2 + (y0 + (q >> 1)) * G.W2 + x0 + (q & 1);
        const int lo = st2[s];
        const int r = s == k2 ? sidx[g] - lo
                              : lower_bound_u32(vals2, lo, en2[s] - lo, (uint32_t)g) - lo;
        rank += tdrop_passes(old2[s], r, G.window);
    }
    const int slot = st3[k3] + rank;
    if (slot < 0 || slot >= *n_dev) return;     // (ranks are a permutation of [0, n))
    keys3[slot] = k3;
    vals3[slot] = (uint32_t)g;
    key3g[g] = k3;
}

// tdrop_s3 over the s3 record order: pass3, the pass-3 list (placed as in
// k_tdrop2; the counters are committed afterwards by k_keys3b) and, for the
// head, each s3 key's last owned pass-3 record (largest record index) and
// their number.
__global__ void __launch_bounds__(256)
k_tdrop3(const int* __restrict__ n_dev, const uint32_t* __restrict__ keys,
         const uint32_t* __restrict__ vals, uint32_t nk, int C, const int* __restrict__ start,
         const int* __restrict__ off, const BlockDesc* __restrict__ bd, int window,
         const unsigned char* __restrict__ owner, int have_head, unsigned char* __restrict__ pass,
         int* __restrict__ list, int* __restrict__ last, int* __restrict__ count) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t k = p < *n_dev ? keys[p] : nk;
    const bool valid = k < nk;
    int g = -1;
    bool own = false;
    if (valid) {
        g = (int)vals[p];
        const int b = (int)k / C, cell = (int)k % C;
        const int r = p - start[k];
        const unsigned c = bd[b].td3[cell];
        const bool take = tdrop_pass(c, (unsigned)r, window);
        pass[g] = take ? 1 : 0;
        if (take) list[off[k] + tdrop_passes(c, r, window)] = g;
        own = take && have_head && owner[g];
    }
    // last / count per key: the records are sorted by key, so a wave holds a
    // few key segments; one lane per segment adds its count and maximum (a
    // per-record atomic put thousands of updates on each of the few keys)
    unsigned long long m = __ballot(own);
    while (m) {
        const uint32_t kl = (uint32_t)__builtin_amdgcn_readlane((int)k, __builtin_ctzll(m));
        const bool in = own && k == kl;
        const unsigned long long sm = __ballot(in);
        int gm = in ? g : -1;
        #pragma unroll
        for (int o = 32; o > 0; o >>= 1) gm = max(gm, __shfl_xor(gm, o));
        if ((threadIdx.x & 63) == __builtin_ctzll(sm)) {
            atomicMax(last + kl, gm);
            atomicAdd(count + kl, __popcll(sm));
        }
        m &= ~sm;
    }
}

// Per s3 key: commit the counter and the pair count of the key.
__global__ void k_keys3b(uint32_t nk3, Geometry G, const int* __restrict__ t3,
                         const BlockDesc* __restrict__ bd, int* __restrict__ pcnt) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nk3) return;
    const int b = (int)t / G.C3, cell = (int)t % G.C3, ty = cell / G.W3, tx = cell % G.W3;
    unsigned char* td = bd[b].td3 + cell;
    *td = (unsigned char)(((unsigned)*td + (unsigned)t3[t]) & 255u);
    int np = 0;
    #pragma unroll
    for (int oy = -1; oy <= 1; ++oy)
        #pragma unroll
        for (int ox = -1; ox <= 1; ++ox) {
            const int sy = ty + oy, sx = tx + ox;
            if (sy < 0 || sy >= G.H3 || sx < 0 || sx >= G.W3) continue;
            np += t3[b * G.C3 + sy * G.W3 + sx];
        }
    pcnt[t] = np;
}

// Pair order without a pair sort.  Pair (record g, delta d) updates the
// patch cell t = (y + 1 - d / 3, x + 1 - d % 3) of g's centre cell (x, y),
// delta = (1 - dy) * 3 + (1 - dx), when t is on the grid.  Pairs are ordered
// by t, and inside t by g: a record adds at most one pair to a cell, so this
// is the stable order of (t, g * 9 + d).  With the records sorted stably by
// centre cell (run [st, en) of ascending record ids per key), t's pair count
// is the sum of the run lengths over its 3 x 3 neighbourhood, and a pair's
// rank inside t is the number of records below g in those nine runs.
//
// One thread per sorted record i (record g = vals[i], key k = keys[i]): the
// ranks of g in the 5 x 5 runs around its centre cell (its own run gives
// i - st[k]), folded row by row into three horizontal 3-sums; a delta's rank
// is the sum of three of them.  The pair's entry at its place in the pair
// order is {9 g + d, t's key}, with kPairNeed set in the id when g needs the
// layer's output (pass[g], or `take` when pass is null: the tdrop decision the
// same thread just made), so k_pscan reads all it needs of a pair in its own
// order.  The lanes of a wave that share a centre cell (records are sorted by
// cell) rank together: every load then serves the whole segment, which keeps
// the L2 request count low.
constexpr uint32_t kPairNeed = 0x80000000u;      // (9 records fit 31 bits)
constexpr int kSegMax = 4;   // cell segments of a wave ranked together; more: per lane
constexpr int kChunkWide = 512;   // widest window counted in 64-value chunks

// r25[c] for the lanes `in` of one segment (lanes l0..l1 holding records of
// key ks, ids ascending): in each neighbour run c of the 5 x 5 block, every
// such lane's lower bound lies between those of lanes l0 and l1, which 48
// lanes find by binary search at once.  The windows are then read 64 values
// at a time, one coalesced load per window (chunk j of every window together),
// and each lane counts the values below its id by a six-step search across
// the lanes (ds_bpermute), the 24 windows' searches interleaved.  Windows
// wider than kChunkWide are searched per lane inside their bounds, all of
// them advanced together.  Every lane of the wave takes part.
__device__ __forceinline__ void
rank_segment(uint32_t ks, int l0, int l1, bool in, uint32_t g, const uint32_t* __restrict__ vals,
             int C, int W, int H, const int* __restrict__ st, const int* __restrict__ en,
             int* r25) {
    const int lane = threadIdx.x & 63;
    const int b = (int)ks / C, cell = (int)ks % C, y = cell / W, x = cell % W;
    const uint32_t g_first = (uint32_t)__builtin_amdgcn_readlane((int)g, l0);
    const uint32_t g_last = (uint32_t)__builtin_amdgcn_readlane((int)g, l1);
    // lanes c and 32 + c (c < 25): run c's bounds for the first and last id
    int bnd = 0, s0 = 0;
    {
        const int c = lane & 31;
        const int sy = y + c / 5 - 2, sx = x + c % 5 - 2;
        if (c < 25 && c != 12 && sy >= 0 && sy < H && sx >= 0 && sx < W) {
            const int s = b * C + sy * W + sx;
            s0 = st[s];
            bnd = lower_bound_u32(vals, s0, en[s] - s0, lane < 32 ? g_first : g_last);
        }
    }
    // windows up to kChunkWide values: read 64 values at a time, one coalesced
    // load per window (chunk j of every window together); each lane counts
    // the values below its id by a six-step search across the lanes
    // (ds_bpermute), the 24 windows' searches interleaved
    int wmax = 0;
    #pragma unroll
    for (int c = 0; c < 25; ++c) {
        const int wa = __builtin_amdgcn_readlane(bnd, c);
        const int we = __builtin_amdgcn_readlane(bnd, 32 + c);
        if (c != 12 && we - wa <= kChunkWide) wmax = max(wmax, we - wa);
    }
    int lo25[25];
    #pragma unroll
    for (int c = 0; c < 25; ++c) lo25[c] = 0;
    for (int base = 0; base < wmax; base += 64) {
        uint32_t pw[25];
        #pragma unroll
        for (int c = 0; c < 25; ++c) {
            const int wa = __builtin_amdgcn_readlane(bnd, c);
            const int we = __builtin_amdgcn_readlane(bnd, 32 + c);
            pw[c] = (c != 12 && we - wa <= kChunkWide && wa + base + lane < we)
                        ? vals[wa + base + lane] : 0xffffffffu;
        }
        int lc[25];
        #pragma unroll
        for (int c = 0; c < 25; ++c) lc[c] = 0;
        #pragma unroll
        for (int step = 32; step > 0; step >>= 1) {
            #pragma unroll
            for (int c = 0; c < 25; ++c) {
                const uint32_t q = (uint32_t)__builtin_amdgcn_ds_bpermute(
                    (lc[c] + step - 1) << 2, (int)pw[c]);
                if (q < g) lc[c] += step;
            }
        }
        #pragma unroll
        for (int c = 0; c < 25; ++c) {
            const uint32_t q = (uint32_t)__builtin_amdgcn_ds_bpermute(lc[c] << 2, (int)pw[c]);
            lo25[c] += lc[c] + (q < g ? 1 : 0);
        }
    }
    // wider still: per-lane binary searches inside the windows, all of them
    // advanced together
    int wlo[25], wlen[25];
    bool wide = false;
    #pragma unroll
    for (int c = 0; c < 25; ++c) {
        const int wa = __builtin_amdgcn_readlane(bnd, c);
        const int we = __builtin_amdgcn_readlane(bnd, 32 + c);
        wlo[c] = wa;
        wlen[c] = (in && c != 12 && we - wa > kChunkWide) ? we - wa : 0;
        wide |= c != 12 && we - wa > kChunkWide;
    }
    if (wide) {
        for (;;) {
            int active = 0;
            #pragma unroll
            for (int c = 0; c < 25; ++c) {
                if (wlen[c] > 0) {
                    const int half = wlen[c] >> 1;
                    if (vals[wlo[c] + half] < g) {
                        wlo[c] += half + 1;
                        wlen[c] -= half + 1;
                    } else {
                        wlen[c] = half;
                    }
                }
                active |= wlen[c];
            }
            if (!active) break;
        }
    }
    #pragma unroll
    for (int c = 0; c < 25; ++c) {
        const int wa = __builtin_amdgcn_readlane(bnd, c);
        const int we = __builtin_amdgcn_readlane(bnd, 32 + c);
        const int ws = __builtin_amdgcn_readlane(s0, c);
        if (in && c != 12) r25[c] = wa - ws + (we - wa > kChunkWide ? wlo[c] - wa : lo25[c]);
    }
}

// A wave's lanes are consecutive records of the sorted order.  When they
// span at most kSegMax keys (the usual case of a large call), each key's segment
// is ranked by rank_segment; otherwise, and always when vals is in LDS (LV: a
// small call, whose runs are short), each lane searches the 24 whole runs, all 24
// binary searches advanced together.
template <bool LV>
__device__ __forceinline__ void
pair_rank_at(int i, int n, const uint32_t* __restrict__ keys,
             const uint32_t* __restrict__ vals, uint32_t nk, int C, int W, int H,
             const int* __restrict__ st, const int* __restrict__ en, const int* __restrict__ pst,
             uint2* __restrict__ pent, const unsigned char* __restrict__ pass, bool take) {
    const int lane = threadIdx.x & 63;
    const bool valid = i < n;
    const uint32_t k = valid ? keys[i] : nk;
    const uint32_t g = valid ? vals[i] : 0u;
    const bool keyed = valid && k < nk;
    const uint32_t kprev = (uint32_t)__builtin_amdgcn_ds_bpermute(((lane + 63) & 63) << 2, (int)k);
    const unsigned long long kmask = __ballot(keyed);
    const int nseg = __popcll(__ballot(keyed && (lane == 0 || kprev != k)));
    // r25[c]: the number of records below g in run c of the 5 x 5 block
    // (c = 5 row + column, c = 12 the record's own run)
    int r25[25];
    #pragma unroll
    for (int c = 0; c < 25; ++c) r25[c] = 0;
    if (!LV && nseg <= kSegMax) {
        unsigned long long left = kmask;
        while (left) {
            const int l0 = (int)__ffsll((long long)left) - 1;
            const uint32_t ks = (uint32_t)__builtin_amdgcn_readlane((int)k, l0);
            const unsigned long long seg = __ballot(keyed && k == ks);
            const int l1 = 63 - (int)__clzll((long long)seg);
            rank_segment(ks, l0, l1, (seg >> lane) & 1ull, g, vals, C, W, H, st, en, r25);
            left &= ~seg;
        }
    } else if (keyed) {
        const int b = (int)k / C, cell = (int)k % C, y = cell / W, x = cell % W;
        int lo[25], len[25];
        #pragma unroll
        for (int c = 0; c < 25; ++c) {
            const int sy = y + c / 5 - 2, sx = x + c % 5 - 2;
            const bool on = c != 12 && sy >= 0 && sy < H && sx >= 0 && sx < W;
            const int s = on ? b * C + sy * W + sx : 0;
            lo[c] = r25[c] = on ? st[s] : 0;
            len[c] = on ? en[s] - lo[c] : 0;
        }
        for (;;) {
            int active = 0;
            #pragma unroll
            for (int c = 0; c < 25; ++c) {
                if (len[c] > 0) {
                    const int half = len[c] >> 1;
                    if (vals[lo[c] + half] < g) {
                        lo[c] += half + 1;
                        len[c] -= half + 1;
                    } else {
                        len[c] = half;
                    }
                }
                active |= len[c];
            }
            if (!active) break;
        }
        #pragma unroll
        for (int c = 0; c < 25; ++c) r25[c] = lo[c] - r25[c];
    }
    if (!keyed) return;
    const int b = (int)k / C, cell = (int)k % C, y = cell / W, x = cell % W;
    const uint32_t need = (pass ? pass[g] != 0 : take) ? kPairNeed : 0u;
    r25[12] = i - st[k];
    int hs[5][3];                  // hs[row][dx + 1]: runs (row, dx - 1 .. dx + 1)
    #pragma unroll
    for (int row = 0; row < 5; ++row)
        #pragma unroll
        for (int c = 0; c < 3; ++c)
            hs[row][c] = r25[5 * row + c] + r25[5 * row + c + 1] + r25[5 * row + c + 2];
    #pragma unroll
    for (int d = 0; d < kPatch; ++d) {
        const int dy = 1 - d / 3, dx = 1 - d % 3;      // target offset from the centre
        const int ty = y + dy, tx = x + dx;
        if (ty < 0 || ty >= H || tx < 0 || tx >= W) continue;
        const int rank = hs[dy + 1][dx + 1] + hs[dy + 2][dx + 1] + hs[dy + 3][dx + 1];
        const int t = b * C + ty * W + tx;
        pent[pst[t] + rank] = make_uint2((g * kPatch + d) | need, (uint32_t)t);
    }
}

// A small call's sorted records in LDS: the searches of a wave are dependent
// loads, and a small call has too few waves to hide them (at 4100 records the s2
// tables took 47 us with the searches in memory).
constexpr int kSmallRec = 8 * kScanThreads;

__device__ __forceinline__ void stage_vals(int n, const uint32_t* __restrict__ vals, uint32_t* sv) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) sv[i] = vals[i];
    __syncthreads();
}

template <bool SMALL>
__global__ void __launch_bounds__(256)
k_pair_rank(int n_max, const int* __restrict__ n_dev, const uint32_t* __restrict__ keys,
            const uint32_t* __restrict__ vals, uint32_t nk, int C, int W, int H,
            const int* __restrict__ st, const int* __restrict__ en, const int* __restrict__ pst,
            uint2* __restrict__ pent, const unsigned char* __restrict__ pass) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, n = n_dev ? *n_dev : n_max;
    if constexpr (SMALL) {
        __shared__ uint32_t sv[kSmallRec];
        if ((int)(blockIdx.x * blockDim.x) >= n) return;
        stage_vals(n, vals, sv);
        pair_rank_at<true>(i, n, keys, sv, nk, C, W, H, st, en, pst, pent, pass, false);
    } else {
        pair_rank_at<false>(i, n, keys, vals, nk, C, W, H, st, en, pst, pent, pass, false);
    }
}

// The s2 level's tables that need only the sorted order and the key scan, in
// one launch: per sorted record (blocks [0, nbr)) its tdrop_s2 decision and
// list slot (tdrop2_at) and its pair ranks; per key (blocks nbr.., when the key
// scan did not build the group list) the groups it leads.
template <bool SMALL>
__global__ void __launch_bounds__(256)
k_s2_tables(int n, int nbr, const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
            uint32_t nk, int C, int W, int H, const int* __restrict__ st,
            const int* __restrict__ en, const int* __restrict__ pst,
            const unsigned char* __restrict__ old,
            const int* __restrict__ off, int window, unsigned char* __restrict__ pass,
            int* __restrict__ list, uint2* __restrict__ pent, int* __restrict__ gcnt,
            int* __restrict__ gend, int* __restrict__ ghist, int* __restrict__ gw) {
    if ((int)blockIdx.x >= nbr) {
        key_group_at((blockIdx.x - (unsigned)nbr) * 256u + threadIdx.x, nk, pst, gcnt, gend, ghist,
                     gw);
        return;
    }
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool take = tdrop2_at(i, n, keys, vals, nk, st, old, off, window, pass, list);
    if constexpr (SMALL) {
        __shared__ uint32_t sv[kSmallRec];
        stage_vals(n, vals, sv);
        pair_rank_at<true>(i, n, keys, sv, nk, C, W, H, st, en, pst, pent, nullptr, take);
    } else {
        pair_rank_at<false>(i, n, keys, vals, nk, C, W, H, st, en, pst, pent, nullptr, take);
    }
}

// ---------------------------------------------------------------------------
// The ordering of a small call (k_small_order): workgroup 0 does, in LDS, what
// k_decode's keys, the radix sort and the key scan do in five launches for
// larger calls (ALL: the pair tables and the whole s3 ordering too, thirteen
// launches); the other workgroups copy the input rows, rebuild the weight copies
// and write the block table.  A small call's launches are latency, not work,
// but one workgroup's work grows with the records: ALL takes 40 us at 300
// records, where the launches it replaces took 110 on the call's critical path,
// and would take 220 at 4100 (the pair ranks 113 of them), so it stops at one
// record per thread; the sort and key tables alone take 27 us at 4100 records
// against about 70, and stop at what the LDS holds (kSmallRec).
// ---------------------------------------------------------------------------
constexpr int kSmallAll = kScanThreads;          // records of an ALL call
constexpr int kSmallGroups = kSmallRec / kGP + 3;
constexpr int kSmallWaves = kScanThreads / 64;

struct SmallOut {
    int* cell2;
    unsigned char *owner, *pass2, *pass3;
    int *list2, *list3, *counts, *last3, *cnt3;
    uint32_t* key3g;
    uint2 *pent2, *pent3;
    int4 *glist2, *glist3;
    int have_head;
    // not ALL: the tables of the launches that follow
    uint32_t *keys2, *vals2;
    int *sidx, *st2, *en2, *pst2, *n2, *off2;
    unsigned char* old2;
};

struct SmallLds {
    uint32_t v2[kSmallRec], k2[kSmallRec];       // records in s2 order, their keys
    unsigned short key[kSmallRec];               // by record: s2 key | owner << 15
    union {
        unsigned short wc[kSmallWaves][kScanThreads + 2];    // sort: counts per wave and key
        struct {
            uint32_t v3[kSmallAll], k3[kSmallAll];           // pass-2 records in s3 order
        };
    };
    int st[kScanThreads + 1], pst[kScanThreads + 1], cur[kScanThreads + 1], go[kScanThreads];
    int n2[kScanThreads], off[kScanThreads];
    unsigned char old[kScanThreads];
    int hist[kSmallGroups], start[kSmallGroups];
    int last[kScanThreads / 4], cnt[kScanThreads / 4];
    int lds[2 * (kScanThreads / 64)];
};
static_assert(sizeof(SmallLds) <= 160 * 1024 - 256, "LDS of the small ordering");

// exclusive scan over the workgroup, one value per thread (k < n): out[k], and
// out[n] = the sum
__device__ __forceinline__ int scan_keys(int v, int n, int* out, int* lds) {
    int total;
    const int k = (int)threadIdx.x, x = block_exscan(k < n ? v : 0, lds, &total);
    if (k < n) out[k] = x;
    if (k == 0) out[n] = total;
    return total;
}

// pairs of key k: the run lengths (st) of its 3 x 3 neighbourhood
__device__ __forceinline__ int pair_count(int k, int C, int W, int H, const int* st) {
    const int b = k / C, cell = k % C, ty = cell / W, tx = cell % W;
    int np = 0;
    #pragma unroll
    for (int oy = -1; oy <= 1; ++oy)
        #pragma unroll
        for (int ox = -1; ox <= 1; ++ox) {
            const int sy = ty + oy, sx = tx + ox;
            if (sy < 0 || sy >= H || sx < 0 || sx >= W) continue;
            const int s = b * C + sy * W + sx;
            np += st[s + 1] - st[s];
        }
    return np;
}

template <bool ALL>
__global__ void __launch_bounds__(kScanThreads)
k_small_order(int E, BlockTable tab, BlockDesc* __restrict__ bd_out, Geometry G,
              float* __restrict__ X0, SmallOut o, PackSrc ps, float* __restrict__ pbuf, int npk) {
    __shared__ SmallLds S;
    const int t = (int)threadIdx.x, wv = t >> 6, lane = t & 63;
    if (blockIdx.x > 0) {
        const int xb = (int)blockIdx.x - 1;
        if (xb < npk) {
            const size_t q = (size_t)xb * kScanThreads + t;
            if (q < PackLayout<true>::off[8]) pack_elem<true>(ps, pbuf, q);
            return;
        }
        // input rows: eight lanes per 128-byte record (as k_decode)
        const int g = (xb - npk) * (kScanThreads / 8) + (t >> 3), c = t & 7;
        if (xb == npk && t < SSLA_MAX_BLOCKS) bd_out[t] = tab.d[t];
        if (g >= E || c < 1 || c > SSLA_C1 / 4) return;
        int b = 0;
        for (int i = 1; i < G.nb; ++i)
            if (g >= tab.d[i].offset) b = i;
        const HybridInputRec* r = tab.d[b].ring + (g - tab.d[b].offset);
        const float4 v = reinterpret_cast<const float4*>(r)[c];
        const bool valid = r->x < G.W2 && r->y < G.H2;
        reinterpret_cast<float4*>(X0 + (size_t)g * SSLA_C1)[c - 1] =
            valid ? v : make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    const int nk2 = G.nb * G.C2, nk3 = G.nb * G.C3, nv = E / kGP + 3;
    const int rounds = (E + kScanThreads - 1) / kScanThreads;
    // ---- keys of the records, their counts -----------------------------------
    for (int i = t; i <= kScanThreads; i += kScanThreads) S.cur[i] = 0;
    for (int i = t; i < kSmallWaves * (kScanThreads + 2); i += kScanThreads) (&S.wc[0][0])[i] = 0;
    if (t < nv) S.hist[t] = 0;
    if (t < 16) o.counts[t] = 0;
    __syncthreads();
    for (int g = t; g < E; g += kScanThreads) {
        int b = 0;
        for (int i = 1; i < G.nb; ++i)
            if (g >= tab.d[i].offset) b = i;
        const HybridInputRec* r = tab.d[b].ring + (g - tab.d[b].offset);
        const HybridStrip& s = tab.d[b].strip;
        const int x = r->x, y = r->y;
        const bool valid = x < G.W2 && y < G.H2;
        const bool own = valid && x >= s.owned_lo && x < s.owned_hi && y >= s.owned_y_lo &&
                         y < s.owned_y_hi;
        const int k = valid ? b * G.C2 + y * G.W2 + x : nk2;
        o.cell2[g] = valid ? y * G.W2 + x : -1;
        o.owner[g] = own ? 1 : 0;
        S.key[g] = (unsigned short)(k | (own ? 0x8000 : 0));
        atomicAdd(&S.cur[k], 1);
    }
    __syncthreads();
    {
        const int len = t < nk2 ? S.cur[t] : 0;
        scan_keys(len, nk2, S.st, S.lds);
        __syncthreads();
        S.cur[t] = t <= nk2 ? S.st[t] : 0;
        if (t == 0) S.cur[kScanThreads] = S.st[nk2];    // (keyless records, nk2 = kScanThreads)
    }
    __syncthreads();
    // ---- stable sort: 1024 records a round, ranks as in k_rs_scatter ------------
    for (int q = 0; q < rounds; ++q) {
        const int g = q * kScanThreads + t;
        const bool valid = g < E;
        const int k = valid ? S.key[g] & 0x7fff : 0;
        unsigned long long peers = __ballot(valid);
        #pragma unroll
        for (int b = 0; b < 11; ++b) {
            const bool bit = (k >> b) & 1;
            const unsigned long long m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const int rank = __popcll(peers & ((1ull << lane) - 1ull)), size = __popcll(peers);
        const bool leader = valid && rank == 0;
        if (leader) S.wc[wv][k] = (unsigned short)size;
        __syncthreads();
        if (valid) {
            int pos = S.cur[k] + rank;
            for (int w = 0; w < wv; ++w) pos += S.wc[w][k];
            S.v2[pos] = (uint32_t)g;
            S.k2[pos] = (uint32_t)k;
            if constexpr (!ALL) {
                o.vals2[pos] = (uint32_t)g;
                o.keys2[pos] = (uint32_t)k;
                o.sidx[g] = pos;
            }
        }
        __syncthreads();
        if (leader) {
            atomicAdd(&S.cur[k], size);
            S.wc[wv][k] = 0;
        }
        __syncthreads();
    }
    // ---- s2 keys: counters, pass-2 counts and offsets, pairs, groups -------------
    {
        int n2 = 0, np = 0;
        if (t < nk2) {
            const int b = t / G.C2, len = S.st[t + 1] - S.st[t];
            unsigned char* td = tab.d[b].td2 + t % G.C2;
            const unsigned c = *td;
            S.old[t] = (unsigned char)c;
            n2 = tdrop_passes(c, len, G.window);
            *td = (unsigned char)((c + (unsigned)len) & 255u);
            S.n2[t] = n2;
            np = pair_count(t, G.C2, G.W2, G.H2, S.st);
        }
        int total;
        const int off = block_exscan(n2, S.lds, &total);
        const int go = block_exscan((np + kGP - 1) / kGP, S.lds, &total);
        if (t < nk2) {
            S.off[t] = off;
            S.go[t] = go;
        }
        if constexpr (!ALL) {
            if (t < nk2) {
                o.st2[t] = S.st[t];
                o.en2[t] = S.st[t + 1];
                o.old2[t] = S.old[t];
                o.n2[t] = n2;
                o.off2[t] = off;
            }
            int n2all;
            (void)block_exscan(n2, S.lds, &n2all);
            if (t == 0) o.counts[0] = n2all;
            if (o.have_head && t < nk3) {
                o.last3[t] = -1;
                o.cnt3[t] = 0;
            }
        }
        scan_keys(np, nk2, S.pst, S.lds);
    }
    __syncthreads();
    if constexpr (!ALL)
        for (int i = t; i <= nk2; i += kScanThreads) o.pst2[i] = S.pst[i];
    group_list_lds(nk2, S.pst, S.go, S.hist, S.start, S.lds, GroupTab{nv, o.glist2, o.counts + 6});
    if constexpr (!ALL) return;
    // ---- one record per thread from here ----------------------------------------
    {
        const bool take = tdrop2_at(t, E, S.k2, S.v2, (uint32_t)nk2, S.st, S.old, S.off, G.window,
                                    o.pass2, o.list2);
        pair_rank_at<true>(t, E, S.k2, S.v2, (uint32_t)nk2, G.C2, G.W2, G.H2, S.st, S.st + 1, S.pst,
                     o.pent2, nullptr, take);
    }
    // ---- s3 keys: run lengths (in cur), starts, pass-3 counts and offsets ---------
    // (the s2 pair starts, offsets and group tables are done with: their arrays
    // take the s3 level's; st, n2, old stay for the s3 ranks)
    __syncthreads();
    {
        int t3 = 0, n3 = 0;
        if (t < nk3) {
            const int b = t / G.C3, cell = t % G.C3;
            const int s = b * G.C2 + 2 * (cell / G.W3) * G.W2 + 2 * (cell % G.W3);
            t3 = S.n2[s] + S.n2[s + 1] + S.n2[s + G.W2] + S.n2[s + G.W2 + 1];
            n3 = tdrop_passes(tab.d[b].td3[cell], t3, G.window);
            S.last[t] = -1;
            S.cnt[t] = 0;
        }
        if (t < nv) S.hist[t] = 0;
        const int n2all = scan_keys(t3, nk3, S.cur, S.lds);
        const int n3all = scan_keys(n3, nk3, S.pst, S.lds);
        if (t < nk3) S.off[t] = S.pst[t];
        if (t == 0) {
            o.counts[0] = n2all;
            o.counts[1] = n3all;
        }
        __syncthreads();
        int np = 0;
        if (t < nk3) np = pair_count(t, G.C3, G.W3, G.H3, S.cur);
        int total;
        const int go = block_exscan((np + kGP - 1) / kGP, S.lds, &total);
        if (t < nk3) S.go[t] = go;
        scan_keys(np, nk3, S.pst, S.lds);
    }
    // the pass-2 records in s3 order (ranks as in k_place3)
    const int k2 = t < E ? (int)S.k2[t] : nk2;
    if (k2 < nk2 && tdrop_pass(S.old[k2], (unsigned)(t - S.st[k2]), G.window)) {
        const int i = t, k = k2;
        const uint32_t g = S.v2[i];
        const int b = k / G.C2, cell = k % G.C2, x = cell % G.W2, y = cell / G.W2;
        const int x0 = x & ~1, y0 = y & ~1;
        const int k3 = b * G.C3 + (y >> 1) * G.W3 + (x >> 1);
        int rank = 0;
        #pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int s = b * G.C2 + (y0 + (q >> 1)) * G.W2 + x0 + (q & 1);
            const int lo = S.st[s];
            const int r = s == k ? i - lo : lower_bound_u32(S.v2, lo, S.st[s + 1] - lo, g) - lo;
            rank += tdrop_passes(S.old[s], r, G.window);
        }
        const int slot = S.cur[k3] + rank;
        if (slot >= 0 && slot < kSmallAll) {              // (ranks are a permutation of [0, n))
            S.k3[slot] = (uint32_t)k3;
            S.v3[slot] = g;
            o.key3g[g] = (uint32_t)k3;
        }
    }
    __syncthreads();
    group_list_lds(nk3, S.pst, S.go, S.hist, S.start, S.lds, GroupTab{nv, o.glist3, o.counts + 7});
    const int n2all = S.cur[nk3];
    {
        const int p = t;
        bool take = false;
        if (p < n2all) {
            const int k = (int)S.k3[p], g = (int)S.v3[p];
            const int r = p - S.cur[k];
            const unsigned c = tab.d[k / G.C3].td3[k % G.C3];
            take = tdrop_pass(c, (unsigned)r, G.window);
            o.pass3[g] = take ? 1 : 0;
            if (take) {
                o.list3[S.off[k] + tdrop_passes(c, r, G.window)] = g;
                if (S.key[g] & 0x8000) {
                    atomicMax(&S.last[k], g);
                    atomicAdd(&S.cnt[k], 1);
                }
            }
        }
        pair_rank_at<true>(p, n2all, S.k3, S.v3, (uint32_t)nk3, G.C3, G.W3, G.H3, S.cur, S.cur + 1, S.pst,
                     o.pent3, nullptr, take);
    }
    __syncthreads();
    if (t < nk3) {
        unsigned char* td = tab.d[t / G.C3].td3 + t % G.C3;
        *td = (unsigned char)(((unsigned)*td + (unsigned)(S.cur[t + 1] - S.cur[t])) & 255u);
        if (o.have_head) {
            o.last3[t] = S.last[t];
            o.cnt3[t] = S.cnt[t];
        }
    }
}

// ---------------------------------------------------------------------------
// P + S: projection and recurrence in one kernel (k_pscan).  Per layer, every
// (record, delta) pair needs v, g = x_record Wvg[delta] and then
// h = sigmoid(g) h + v along its cell's pairs in ring order.  A workgroup (one
// per CU, 16 waves, persistent) takes groups of up to kGP pairs of the pair
// order (see key_groups) and 48 of the layer's channels at a time; its waves
// have roles and hand groups on through LDS counters (PsSlot), with up to four
// groups in flight:
//   deal (1 wave)   draws tickets two ahead, loads a group's pairs and deals
//     them into 16-pair MFMA tiles of one delta each (a tile's missing pairs
//     repeat a record and write a spare row);
//   tiles (8 waves, two per SIMD)   per tile the records' input rows are the B
//     operand (one float4 per lane and four k-steps, straight from the feature
//     rows, the next tile's while a tile runs) and the delta's weights the A
//     operand (fragment order, ProjPackT, streamed DW - 1 parts ahead), so a
//     lane's four results are four channels of one pair: v and sigmoid(g) go to
//     the pair's row in LDS.  The [v | g] rows never reach memory;
//   rows (two teams of 3 waves, every other group each)   thread (sub, channel)
//     takes kPSRows consecutive rows into registers, which frees the LDS buffer
//     for the group after the next, and composes their map h -> A h + B (a cell's
//     first pair has its cell's stored state folded in and drops what came
//     before); with its start state it replays them, writes h at row 9 g + d where
//     the pair's record needs the layer's output (a record's nine rows are
//     contiguous for its contraction), and stores the state of a cell's last pair;
//   chain (1 wave)   composes the group's map and finds its start state: none
//     needed for a group that begins with a cell's first pair, else by looking
//     back over the cell's earlier groups -- the nearest one whose end state is
//     published, then the maps of the groups after it, applied forward.  A group
//     publishes its map before it waits and its end state once it has its start,
//     so every state is the same fixed chain of fmaf's whichever word a reader
//     happens to find: the results do not depend on timing.
// Tickets: group_order lists a group's predecessors in its cell before it.  A
// workgroup holds several tickets, works on them in ascending order and waits
// only for smaller ones, so the smallest unfinished ticket never waits.
// Published words hold a float and the launch's tag (value | tag << 32) and are
// stored and loaded with relaxed device-scope atomics: a reader that sees the
// tag sees the value, with no fence (a release fence would write back the L2).
// Every wait on another workgroup is bounded on the wall clock; a wave that runs
// out raises *err (host memory) and goes on with a zero state.
//
// Bounds and measurements (200k records at 80 x 64, L4 / L5 / L6 / L7): the fp32
// matrix cores need 67 / 135 / 62 / 127 us for the tiles (11 pairs of a tile's 16
// are real: 9 deltas share a group's 176 pairs), and are busy 35 / 50 / 42 / 54% of
// 0.21 / 0.30 / 0.157 / 0.25 ms.  The two launches this replaced (projection to pair
// rows in memory, one-pass scan over them) took 0.41 / 0.38 / 0.22 / 0.26 ms; a call
// moved 6.0 GB and moves 2.4, and went from 1.80 to 1.43 ms.  Loads are not the
// bound (rows or weights from the L1 changed the times by 2-8%).  Measured on the
// way, in ms per call beside 1.40 for the kept form in the same runs: workgroups of
// 6 waves do not pair on a CU (2.05); 8 waves that run all phases in turn, two
// workgroups per CU, 1.70; the same with look-back and replay of a group behind the
// tiles of the next, 1.52; one row team of 3 waves and 11 tile waves, 1.51; two
// interleaved accumulator chains per tile wave, 1.43 (a single dependent chain
// forwards its accumulator).
// ---------------------------------------------------------------------------
constexpr int kTM = 64;     // records per head workgroup

// Row stride of the LDS tiles read as MFMA A operands, a[(16 m + li) ST + lk
// + 4 s] with li = lane % 16, lk = lane / 16: a stride of 2 (mod 4) puts the
// 32 lanes of each half-wave on 32 distinct banks (a multiple of 4 pairs row
// li with row li + 8).  Rows are then 8-byte aligned: written as float2.
constexpr int lds_stride(int n) { return n + 2; }    // n % 4 == 0

__device__ __forceinline__ void lds_put4(float* p, float4 v) {
    reinterpret_cast<float2*>(p)[0] = make_float2(v.x, v.y);
    reinterpret_cast<float2*>(p)[1] = make_float2(v.z, v.w);
}

constexpr int kLB = 4;       // groups looked at per look-back step

__device__ __forceinline__ void sw_put(unsigned long long* p, float v, unsigned tag) {
    __hip_atomic_store(p, ((unsigned long long)tag << 32) | __float_as_uint(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long sw_get(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool sw_ok(unsigned long long x, unsigned tag) {
    return (unsigned)(x >> 32) == tag;
}
__device__ __forceinline__ float sw_val(unsigned long long x) {
    return __uint_as_float((unsigned)x);
}

// Start state of the group of rank r > 0 of a cell (channel cc of a lane;
// `on` marks the lanes that carry a channel).  The cell's group of rank x
// publishes [end | SA | SB] x OUT words at sw + (slot0 + x) 3 OUT; rank 0
// publishes its end state without waiting.
template <int OUT>
__device__ float scan_lookback(const unsigned long long* __restrict__ sw, int slot0, int r, int cc,
                               bool on, unsigned tag, unsigned long long deadline,
                               int* __restrict__ err) {
    auto word = [&](int x) { return sw + ((size_t)slot0 + (size_t)x) * 3 * OUT + cc; };
    // phase 1: the nearest group whose end state every lane sees
    int top = r - 1, found = -1;
    float h = 0.f;
    for (;;) {
        unsigned long long x[kLB];
        #pragma unroll
        for (int q = 0; q < kLB; ++q) x[q] = sw_get(word(max(top - q, 0)));
        #pragma unroll
        for (int q = 0; q < kLB; ++q) {
            const bool ok = top - q >= 0 && __all(!on || sw_ok(x[q], tag));
            if (found < 0 && ok) {
                found = top - q;
                h = sw_val(x[q]);
            }
        }
        if (found >= 0) break;
        if (top - kLB >= 0) {
            top -= kLB;                       // none of these: look further back
            continue;
        }
        if ((unsigned long long)wall_clock64() > deadline) {
            if ((threadIdx.x & 63) == 0)
                __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return 0.f;
        }
        __builtin_amdgcn_s_sleep(2);
        top = r - 1;                          // start again from the nearest group
    }
    // phase 2: the maps of the groups after it, applied forward
    for (int x0 = found + 1; x0 < r; x0 += kLB) {
        unsigned long long a[kLB], b[kLB];
        for (;;) {
            #pragma unroll
            for (int q = 0; q < kLB; ++q) {
                const unsigned long long* p = word(min(x0 + q, r - 1));
                a[q] = sw_get(p + OUT);
                b[q] = sw_get(p + 2 * OUT);
            }
            bool ok = true;
            #pragma unroll
            for (int q = 0; q < kLB; ++q) ok = ok && (x0 + q >= r || (sw_ok(a[q], tag) && sw_ok(b[q], tag)));
            if (__all(!on || ok)) break;
            if ((unsigned long long)wall_clock64() > deadline) {
                if ((threadIdx.x & 63) == 0)
                    __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                return 0.f;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        #pragma unroll
        for (int q = 0; q < kLB; ++q)
            if (x0 + q < r) h = fmaf(sw_val(a[q]), h, sw_val(b[q]));
    }
    return h;
}

constexpr int kPSC = 48;                    // channels per workgroup
constexpr int kPSTileWaves = 8;             // waves 0..7: tiles (two per SIMD)
constexpr int kPSTeam = 3;                  // waves 8..10: rows of the even groups, 11..13: odd
constexpr int kPSScanWaves = 2 * kPSTeam;
constexpr int kPSDeal = kPSTileWaves + kPSScanWaves;         // wave 14: deals groups
constexpr int kPSChain = kPSDeal + 1;                        // wave 15: start states
constexpr int kPSThreads = 64 * (kPSChain + 1);
constexpr int kPSSub = 64 * kPSTeam / kPSC;                  // row blocks of the scan
constexpr int kPSRows = kGP / kPSSub;                        // rows of a thread
constexpr int kPSStride = 2 * kPSC + 4;     // LDS row [v | sigmoid(g)]: 16 rows on 16 bank groups
constexpr int kPSTiles = kPatch + (kGP - kPatch) / 16;       // most tiles of a group
constexpr int kPSMask = (kGP + 63) / 64;    // 64-pair blocks of a group
constexpr int kPSSlots = 4;                 // groups in flight in a workgroup
constexpr float kPSFirst = -1.f;            // in place of a first row's sigmoid (>= 0 or NaN)
static_assert(kPSSub * kPSC == 64 * kPSTeam && kGP % kPSSub == 0 && kPSRows < 64 &&
                  kGP < 256 && 2 * kGW <= kGP, "group shape");

// One group on its way through a workgroup.
struct PsSlot {
    float* srow[kGP];               // state row of a pair's cell (groups with a cell end)
    unsigned long long mfirst[kPSMask], mlast[kPSMask], mneed[kPSMask];
    int ids[kGP];                   // 9 record + delta
    alignas(4) unsigned char tsl[kPSTiles * 16];        // pairs of each tile
    unsigned char tdel[kPSTiles];                       // its delta
    int ntiles, n, flags, word, r, slab;
    int taken;                      // tiles taken
    // arrivals over all groups that had the slot (a wave reaches the slot's next
    // group only after all have passed this one): tile waves that have left the
    // group, scan waves that have read T, written their maps and replayed
    int left, read, mapped, replayed;
};

// kPSRows bits from bit i of a mask of kPSMask words
__device__ __forceinline__ unsigned long long mask_window(const unsigned long long* m, int i) {
    const int w = i >> 6, o = i & 63;
    unsigned long long x = m[w] >> o;
    if (o > 64 - kPSRows && w + 1 < kPSMask) x |= m[w + 1] << (64 - o);
    return x & ((1ull << kPSRows) - 1ull);
}

// Hand-over between a workgroup's waves by counters in LDS: what a wave wrote
// to LDS before it arrives is seen by a wave that waited for the count.
__device__ __forceinline__ int lds_get(const int* p) {
    return __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}
__device__ __forceinline__ void lds_arrive(int* p) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if ((threadIdx.x & 63) == 0)
        __hip_atomic_fetch_add(p, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_wait(const int* p, int v) {
    while (lds_get(p) < v) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

template <int IN, int OUT, bool ALL, bool NT>
__global__ void __launch_bounds__(kPSThreads, 4)
k_pscan(const int* __restrict__ n_groups, int* __restrict__ ticket, unsigned tag,
        const int4* __restrict__ glist, const uint2* __restrict__ pent, const float* __restrict__ X,
        const float* __restrict__ pp, int C, const BlockDesc* __restrict__ bd, int li,
        float* __restrict__ Hout, unsigned long long* __restrict__ sw, int* __restrict__ err,
        unsigned long long wait_ticks) {
    using P = ProjPackT<IN, OUT>;
    constexpr int KG = P::KG, NS = OUT / kPSC, NJ = 2 * kPSC / 16;
    __shared__ __align__(16) float T[2][(kGP + 1) * kPSStride];   // row kGP: the spare row
    __shared__ PsSlot slot[kPSSlots];
    __shared__ float sA[2][kPSSub][kPSC], sB[2][kPSSub][kPSC];    // sA: then the start states
    __shared__ int dcnt[kPatch];
    // groups dealt, the workgroup's groups (once known), groups with start states
    __shared__ int dealt, n_mine, starts;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (threadIdx.x == 0) {
        dealt = starts = 0;
        n_mine = 0x7fffffff;
    }
    if (threadIdx.x < kPSSlots) {
        PsSlot& S = slot[threadIdx.x];
        S.left = S.read = S.mapped = S.replayed = 0;
    }
    __syncthreads();
    // arrivals of all `waves` in group g's slot, up to and with group g
    auto count = [](int waves, int g) { return waves * (g / kPSSlots + 1); };
    // waits for group g to be dealt; false: the workgroup has no such group
    auto have_group = [&](int g) {
        for (;;) {
            if (lds_get(&dealt) > g) break;
            if (lds_get(&n_mine) <= g) return false;
            __builtin_amdgcn_s_sleep(1);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        return true;
    };

    // the few instructions of the other waves go ahead of the tiles' streams
    if (wv >= kPSDeal) __builtin_amdgcn_s_setprio(3);
    else if (wv >= kPSTileWaves) __builtin_amdgcn_s_setprio(2);
    if (wv < kPSTileWaves) {
        // ---- tiles: v, sigmoid(g) of 16 pairs of one delta --------------------
        // weights are loaded one float4 group (a part, four k-steps) at a time,
        // DW - 1 parts ahead, and the next tile's input rows while a tile runs
        constexpr int NQ = NJ * KG, DW = KG == 2 ? 4 : 6;
        static_assert(NQ % DW == 0 && NQ >= 8, "weight ring");
        const int lc = lane & 15, lk = lane >> 4;
        f32x4 xb[KG], xn[KG], wb[DW];
        auto load_x = [&](int id, f32x4 (&x)[KG]) {
            const float* xp = X + (size_t)((unsigned)id / (unsigned)kPatch) * IN;
            #pragma unroll
            for (int g = 0; g < KG; ++g) {
                if (P::steps(g) == 4) {
                    x[g] = *(const SSLA_GLOBAL f32x4*)(xp + P::kidx(g, lk, 0));
                } else {
                    const f32x2 v = *(const SSLA_GLOBAL f32x2*)(xp + P::kidx(g, lk, 0));
                    x[g] = f32x4{v[0], v[1], 0.f, 0.f};
                }
            }
        };
        // part q of a tile: group q % KG of item q / KG (ds = delta, slab)
        auto load_w = [&](int ds, int q, f32x4& w) {
            const SSLA_GLOBAL f32x4* src = (const SSLA_GLOBAL f32x4*)pp + (size_t)(ds * NQ + q) * 64;
            if (P::steps(q % KG) == 4) {
                w = src[(unsigned)lane];
            } else {
                const f32x2 v = *(const SSLA_GLOBAL f32x2*)(src + (unsigned)lane);
                w = f32x4{v[0], v[1], 0.f, 0.f};
            }
        };
        auto take = [&](PsSlot& S) { return lane == 0 ? atomicAdd(&S.taken, 1) : 0; };
        for (int g = 0; have_group(g);) {
            PsSlot* S = &slot[g % kPSSlots];
            int nt = __builtin_amdgcn_readfirstlane(S->ntiles);
            int tile = __builtin_amdgcn_readfirstlane(take(*S));
            if (tile >= nt) {
                lds_arrive(&S->left);
                ++g;
                continue;
            }
            int lp = S->tsl[tile * 16 + lc];
            int ds = __builtin_amdgcn_readfirstlane(S->tdel[tile] * NS + S->slab);
            load_x(S->ids[lp < kGP ? lp : 0], xb);
            #pragma unroll
            for (int q = 0; q < DW - 1; ++q) load_w(ds, q, wb[q]);
            for (;;) {
                // T[g % 2] is free once group g - 2 has been read
                if (g > 1) lds_wait(&slot[(g - 2) % kPSSlots].read, count(kPSTeam, g - 2));
                float* row = &T[g & 1][lp * kPSStride + 4 * lk];
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                // the next tile, of this group or, if it is dealt, the next one
                // (none: this tile again, so that the loads carry no branch);
                // its look-ups are spread over the first parts
                PsSlot* SN = S;
                int tn = 0, lpn = 0, idn = 0, dsn = 0, gn = g;
                bool more = true;
                #pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    const int j = q / KG, kg = q % KG;
                    if (q == 0) tn = take(*S);
                    if (q == 1) {
                        tn = __builtin_amdgcn_readfirstlane(tn);
                        if (tn >= nt) {
                            gn = g + 1;
                            more = lds_get(&dealt) > gn;
                            if (more) {
                                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                                SN = &slot[gn % kPSSlots];
                                tn = __builtin_amdgcn_readfirstlane(take(*SN));
                                more = tn < __builtin_amdgcn_readfirstlane(SN->ntiles);
                            }
                            if (!more) tn = 0;
                        }
                        lpn = SN->tsl[tn * 16 + lc];
                        dsn = SN->tdel[tn] * NS + SN->slab;
                    }
                    if (q == 2) idn = SN->ids[lpn < kGP ? lpn : 0];
                    if (q == 3) load_x(idn, xn);
                    if (q == NQ - DW + 1) dsn = __builtin_amdgcn_readfirstlane(dsn);
                    if (q + DW - 1 < NQ) load_w(ds, q + DW - 1, wb[(q + DW - 1) % DW]);
                    else load_w(dsn, q + DW - 1 - NQ, wb[(q + DW - 1) % DW]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (kg == 0) acc = f32x4{0.f, 0.f, 0.f, 0.f};
                    #pragma unroll
                    for (int i = 0; i < P::steps(kg); ++i)
                        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wb[q % DW][i], xb[kg][i], acc, 0, 0, 0);
                    if (kg == KG - 1) {
                        if (j >= NJ / 2) {
                            #pragma unroll
                            for (int i = 0; i < 4; ++i) acc[i] = sigmoid_fast(acc[i]);
                        }
                        *reinterpret_cast<f32x4*>(row + 16 * j) = acc;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (gn != g) {
                    lds_arrive(&S->left);
                    g = gn;
                    if (!more) {
                        // (a tile counter taken past its end is harmless)
                        break;
                    }
                    S = SN;
                    nt = __builtin_amdgcn_readfirstlane(S->ntiles);
                }
                lp = lpn;
                ds = dsn;
                #pragma unroll
                for (int k = 0; k < KG; ++k) xb[k] = xn[k];
            }
        }
    } else if (wv < kPSDeal) {
        // ---- rows: maps, replay (two teams, every other group each) --------------
        const int team = (wv - kPSTileWaves) / kPSTeam;
        const int ct = (int)threadIdx.x - 64 * (kPSTileWaves + team * kPSTeam);
        const int sub = ct / kPSC, ch = ct - sub * kPSC, i0 = sub * kPSRows;
        for (int g = team; have_group(g); g += 2) {
            PsSlot& S = slot[g % kPSSlots];
            float vv[kPSRows], ss[kPSRows];
            lds_wait(&S.left, count(kPSTileWaves, g));
            const float* row = &T[g & 1][i0 * kPSStride + ch];
            #pragma unroll
            for (int q = 0; q < kPSRows; ++q) {
                vv[q] = row[q * kPSStride];
                ss[q] = row[q * kPSStride + kPSC];
            }
            lds_arrive(&S.read);
            const int n = __builtin_amdgcn_readfirstlane(S.n);
            const int flags = __builtin_amdgcn_readfirstlane(S.flags);
            if (n < kGP) {
                // rows past the group's pairs leave a state as it is
                #pragma unroll
                for (int q = 0; q < kPSRows; ++q) {
                    vv[q] = i0 + q < n ? vv[q] : 0.f;
                    ss[q] = i0 + q < n ? ss[q] : 1.f;
                }
            }
            // a cell's first row: its state is vv, whatever came before.  A group
            // of one cell has it on top, where the state is 0; in a group of
            // several a product with 0 would let the previous cell's infinity or
            // NaN through, so the row is marked and its state selected (two more
            // instructions a row: 200k records at 80 x 64 1.438 -> 1.439 ms, 1.25 M
            // at 640 x 480 9.23 -> 9.28).
            const bool multi = (flags & kGMulti) != 0;
            if (flags & kGStart) {
                const unsigned long long fw = mask_window(S.mfirst, i0);
                #pragma unroll
                for (int q = 0; q < kPSRows; ++q)
                    if ((fw >> q) & 1u) {
                        vv[q] = fmaf(ss[q], gload(S.srow[i0 + q] + ch), vv[q]);
                        ss[q] = multi ? kPSFirst : 0.f;
                    }
            }
            float A = 1.f, B = 0.f;
            if (multi) {
                // (A is read of row blocks without a first row only)
                #pragma unroll
                for (int q = 0; q < kPSRows; ++q) {
                    A *= ss[q];
                    B = ss[q] == kPSFirst ? vv[q] : fmaf(ss[q], B, vv[q]);
                }
            } else {
                #pragma unroll
                for (int q = 0; q < kPSRows; ++q) {
                    A *= ss[q];
                    B = fmaf(ss[q], B, vv[q]);
                }
            }
            sA[g & 1][sub][ch] = A;
            sB[g & 1][sub][ch] = B;
            lds_arrive(&S.mapped);
            lds_wait(&starts, g + 1);
            float h = sA[g & 1][sub][ch];
            // (one loop for both kinds of group: a second copy spills 29 registers)
            #pragma unroll
            for (int q = 0; q < kPSRows; ++q) {
                h = ss[q] == kPSFirst ? vv[q] : fmaf(ss[q], h, vv[q]);
                vv[q] = h;
            }
            float* const hb = Hout + __builtin_amdgcn_readfirstlane(S.slab) * kPSC + ch;
            auto put = [&](int q) {
                float* hp = hb + (size_t)(unsigned)S.ids[i0 + q] * OUT;
                if constexpr (NT) __builtin_nontemporal_store(vv[q], (SSLA_GLOBAL float*)hp);
                else gstore(hp, vv[q]);
            };
            if (ALL && n == kGP) {
                #pragma unroll
                for (int q = 0; q < kPSRows; ++q) put(q);
            } else {
                const unsigned long long nw =
                    ALL ? (1ull << max(0, min(kPSRows, n - i0))) - 1ull : mask_window(S.mneed, i0);
                #pragma unroll
                for (int q = 0; q < kPSRows; ++q)
                    if ((nw >> q) & 1u) put(q);
            }
            if (flags & kGEnd) {
                const unsigned long long lw = mask_window(S.mlast, i0);
                #pragma unroll
                for (int q = 0; q < kPSRows; ++q)
                    if ((lw >> q) & 1u) gstore(S.srow[i0 + q] + ch, vv[q]);
            }
            lds_arrive(&S.replayed);
        }
    } else if (wv == kPSDeal) {
        // ---- deals the pairs of the next groups into tiles of one delta -----------
        const int total = *n_groups * NS;
        auto draw = [&]() { return lane == 0 ? atomicAdd(ticket, 1) : 0; };
        auto fetch = [&](int tk) { return tk < total ? glist[tk / NS] : make_int4(0, 0, 0, 0); };
        uint2 e[kPSMask];
        auto load_pairs = [&](int4 gd) {
            const int n = gd.y & 0xffff;
            #pragma unroll
            for (int j = 0; j < kPSMask; ++j) {
                e[j] = make_uint2(0u, 0u);
                if (64 * j + lane < n) e[j] = pent[gd.x + 64 * j + lane];
            }
        };
        // in flight: the next group's pairs, the group after it, the ticket after that
        int d0 = 0, d1 = 0, tk2 = 0;
        if (lane == 0) {
            d0 = atomicAdd(ticket, 1);
            d1 = atomicAdd(ticket, 1);
            tk2 = atomicAdd(ticket, 1);
        }
        int tk = __builtin_amdgcn_readfirstlane(d0), tk1 = __builtin_amdgcn_readfirstlane(d1);
        int4 gd = fetch(tk), gd1 = fetch(tk1);
        load_pairs(gd);
        for (int g = 0;; ++g) {
            if (tk >= total) {
                if (lane == 0) __hip_atomic_store(&n_mine, g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                break;
            }
            uint2 ec[kPSMask];
            #pragma unroll
            for (int j = 0; j < kPSMask; ++j) ec[j] = e[j];
            load_pairs(gd1);
            const int t2 = __builtin_amdgcn_readfirstlane(tk2);
            const int4 gd2 = fetch(t2);
            tk2 = draw();
            // the slot is free once group g - kPSSlots has been replayed
            PsSlot& S = slot[g % kPSSlots];
            if (g >= kPSSlots) lds_wait(&S.replayed, count(kPSTeam, g - kPSSlots));
            const int flags = __builtin_amdgcn_readfirstlane(gd.y), n = flags & 0xffff;
            const int slab = NS == 1 ? 0 : tk % NS;
            if (lane < kPatch) dcnt[lane] = 0;
            for (int i = lane; i < kPSTiles * 16 / 4; i += 64)
                reinterpret_cast<uint32_t*>(S.tsl)[i] = kGP * 0x01010101u;
            int rank[kPSMask], delta[kPSMask];
            #pragma unroll
            for (int j = 0; j < kPSMask; ++j) {
                const bool on = 64 * j + lane < n;
                delta[j] = (int)((ec[j].x & ~kPairNeed) % (unsigned)kPatch);
                rank[j] = on ? atomicAdd(&dcnt[delta[j]], 1) : 0;
            }
            // a cell's first and last pairs
            #pragma unroll
            for (int j = 0; j < kPSMask; ++j) {
                const int i = 64 * j + lane;
                bool first = false, last = false;
                if (flags & kGMulti) {
                    uint32_t up = (uint32_t)__shfl_up((int)ec[j].y, 1);
                    uint32_t dn = (uint32_t)__shfl_down((int)ec[j].y, 1);
                    const uint32_t pe = (uint32_t)__builtin_amdgcn_readlane((int)ec[j ? j - 1 : 0].y, 63);
                    const uint32_t ns = (uint32_t)__builtin_amdgcn_readlane(
                        (int)ec[j + 1 < kPSMask ? j + 1 : j].y, 0);
                    if (lane == 0) up = pe;
                    if (lane == 63) dn = ns;
                    first = up != ec[j].y;
                    last = dn != ec[j].y;
                }
                const unsigned long long mf = __ballot(i < n && (i == 0 ? (flags & kGStart) != 0 : first));
                const unsigned long long ml = __ballot(i < n && (i == n - 1 ? (flags & kGEnd) != 0 : last));
                const unsigned long long mn = __ballot(i < n && (ec[j].x & kPairNeed));
                if (lane == 0) {
                    S.mfirst[j] = mf;
                    S.mlast[j] = ml;
                    S.mneed[j] = mn;
                }
            }
            int base[kPSMask] = {}, nt = 0;
            #pragma unroll
            for (int d = 0; d < kPatch; ++d) {
                #pragma unroll
                for (int j = 0; j < kPSMask; ++j)
                    if (delta[j] == d) base[j] = nt;
                nt += (dcnt[d] + 15) >> 4;
            }
            #pragma unroll
            for (int j = 0; j < kPSMask; ++j) {
                const int i = 64 * j + lane;
                if (i < n) {
                    S.tsl[base[j] * 16 + rank[j]] = (unsigned char)i;
                    if ((rank[j] & 15) == 0) S.tdel[base[j] + (rank[j] >> 4)] = (unsigned char)delta[j];
                    S.ids[i] = (int)(ec[j].x & ~kPairNeed);
                    if (flags & (kGStart | kGEnd)) {
                        const int k = (int)ec[j].y, b = k / C;
                        S.srow[i] = bd[b].hidden[li] + (size_t)(k - b * C) * OUT + slab * kPSC;
                    }
                }
            }
            if (lane == 0) {
                S.ntiles = nt;
                S.n = n;
                S.flags = flags;
                S.word = gd.z;
                S.r = gd.w;
                S.slab = slab;
                S.taken = 0;
            }
            lds_arrive(&dealt);
            tk = tk1;
            tk1 = t2;
            gd = gd1;
            gd1 = gd2;
        }
    } else {
        // ---- the groups' maps and start states -----------------------------------
        const bool con = lane < kPSC;
        const int cl = con ? lane : 0;
        for (int g = 0; have_group(g); ++g) {
            const PsSlot& S = slot[g % kPSSlots];
            lds_wait(&S.mapped, count(kPSTeam, g));
            const int flags = __builtin_amdgcn_readfirstlane(S.flags);
            const int word = __builtin_amdgcn_readfirstlane(S.word);
            const int r = __builtin_amdgcn_readfirstlane(S.r);
            const int cc = __builtin_amdgcn_readfirstlane(S.slab) * kPSC + cl;
            // (of a group of several cells only the start states are used: a row
            // block that holds a cell's first row ends in a state of its own)
            float a[kPSSub], b[kPSSub], SA = 1.f, SB = 0.f;
            bool own[kPSSub] = {};
            #pragma unroll
            for (int q = 0; q < kPSSub; ++q) {
                a[q] = sA[g & 1][q][cl];
                b[q] = sB[g & 1][q][cl];
                if (flags & kGMulti) own[q] = mask_window(S.mfirst, q * kPSRows) != 0;
            }
            #pragma unroll
            for (int q = 0; q < kPSSub; ++q) {
                SB = fmaf(a[q], SB, b[q]);
                SA *= a[q];
            }
            unsigned long long* W = sw + (size_t)word * 3 * OUT + cc;
            float h = 0.f;
            if (flags & kGStart) {
                if (!(flags & kGEnd) && con) sw_put(W, SB, tag);       // SA = 0: no start state
            } else {
                if (!(flags & kGEnd) && con) {
                    sw_put(W + OUT, SA, tag);
                    sw_put(W + 2 * OUT, SB, tag);
                }
                h = scan_lookback<OUT>(sw, word - r, r, cc, con, tag,
                                       (unsigned long long)wall_clock64() + wait_ticks, err);
                if (!(flags & kGEnd) && con) sw_put(W, fmaf(SA, h, SB), tag);
            }
            #pragma unroll
            for (int q = 0; q < kPSSub; ++q) {
                if (con) sA[g & 1][q][cl] = h;
                h = own[q] ? b[q] : fmaf(a[q], h, b[q]);
            }
            lds_arrive(&starts);
        }
    }
}

// ---------------------------------------------------------------------------
// O: per record y = sum_delta goW[delta]^T (q_delta * h_delta) + residual,
// fp64 LayerNorm -- computed transposed, with the weights as MFMA A operands
// and the records as columns (layouts in mfma_pack.h, OutPackT):
//   q^T tile (16 channels x 16 records) = Wq[delta]^T X^T
//   Y^T     += goW[delta]^T (q^T * h^T)        for every output tile
//   Y^T     += input_proj^T X^T (IN != OUT) or + X (IN == OUT)
// Each wave owns RT tiles of 16 records and runs every K part itself, so no
// LDS and no barrier are involved: a lane keeps its record's input row
// (the B operand of q and input_proj, one float4 per four steps) in
// registers for the whole kernel; the h values arrive as one float4 per
// lane in the MFMA output layout of the q tile and are multiplied there;
// and with the K order of OutPackT those four products are the lane's B
// values of the goW steps.  The weights stream from the L2 (shared by all
// waves) one (delta, channel tile) item ahead.  LayerNorm in fp64 over the
// four lanes that hold a record's outputs (ds_swizzle and ds_bpermute sums).
// HR holds the h row of pair (record g, delta d) at 9 g + d; whether the pair
// exists follows from g's centre cell (s2 coordinates >> shift, on a W x H grid).
// WPS asks the compiler for at least that many waves per SIMD; with the
// unrolled item loop L4 (RT = 2) compiles to 120 registers, 4 waves per SIMD.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double xor_lanes_d(double v, int pattern_or_lane, bool swizzle) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    unsigned lo, hi;
    if (swizzle) {
        lo = (unsigned)__builtin_amdgcn_ds_swizzle((int)(unsigned)b, 0x401F);       // xor 16
        hi = (unsigned)__builtin_amdgcn_ds_swizzle((int)(unsigned)(b >> 32), 0x401F);
    } else {
        lo = (unsigned)__builtin_amdgcn_ds_bpermute(pattern_or_lane, (int)(unsigned)b);
        hi = (unsigned)__builtin_amdgcn_ds_bpermute(pattern_or_lane, (int)(unsigned)(b >> 32));
    }
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// sum over lanes j, j + 16, j + 32, j + 48 (all 64 lanes active)
__device__ __forceinline__ double sum4_lanes(double v, int lane) {
    v += xor_lanes_d(v, 0, true);
    return v + xor_lanes_d(v, (lane ^ 32) << 2, false);
}

// L5-L7 contraction launch shape: 16-record tiles (RT = 1), the nine deltas
// split over three waves (KS = 3).  Measured at 200k records: nine waves per
// tile (one delta each) took L5.out 61 -> 91 us and L6.out 146 -> 214 us
// (L7 spills at the 168-register cap of nine waves); two record tiles per
// wave left L5.out unchanged and took L6.out to 161 us (L7: 202 registers,
// one wave per SIMD).
constexpr int kOutKS5 = 3, kOutKS6 = 3, kOutKS7 = 3;
constexpr int kOutRT5 = 1, kOutRT6 = 1, kOutRT7 = 1;
// A layer with at most two 16-record tiles per CU is a chain of load latencies
// (27 items a wave in L4), so every delta gets a wave of its own (KS = 9); L7
// keeps three, nine would spill.  At 300 records L4 22 -> 8 us, L6 18 -> 17.
constexpr int kOutKSFew = 9, kOutKSFew7 = 3;

template <int IN, int OUT, int RT, int KS, int WPS = 1>
__global__ void __launch_bounds__(64 * KS, WPS)
k_outt(int n_max, const int* __restrict__ n_dev, const int* __restrict__ list,
       const float* __restrict__ X, const int* __restrict__ cell2, int shift, int W2, int W, int H,
       const float* __restrict__ HR,
       const float* __restrict__ po, const float* __restrict__ gamma,
       const float* __restrict__ beta, float* __restrict__ Y) {
    using O = OutPackT<IN, OUT>;
    constexpr int NT = O::NT, KG = O::KG, R = 16 * RT;
    // the workgroup's pair rows, and the partial sums of waves 1..KS-1
    __shared__ int sp[R][kPatch];
    __shared__ f32x4 part[KS > 1 ? KS - 1 : 1][RT * NT][64];
    const int n = n_dev ? *n_dev : n_max;
    const int base = blockIdx.x * R;
    if (base >= n) return;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
    for (int t = threadIdx.x; t < R * kPatch; t += 64 * KS) {
        const int r = t / kPatch, d = t - r * kPatch;
        const int q = base + r;
        const int rr = q < n ? (list ? list[q] : q) : -1;
        const int cell = rr >= 0 ? cell2[rr] : -1;
        const int tx = ((cell % W2) >> shift) + 1 - d % 3, ty = ((cell / W2) >> shift) + 1 - d / 3;
        sp[r][d] = cell >= 0 && tx >= 0 && tx < W && ty >= 0 && ty < H ? rr * kPatch + d : -1;
    }
    int rec[RT];
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int r = base + 16 * rt + j;
        rec[rt] = r < n ? (list ? list[r] : r) : -1;
    }
    // this lane's B values of the input steps: X[rec][16 t + 4 g .. + 3]
    // (a half group: X[rec][16 t + 2 g .. + 1])
    f32x4 xr[RT][KG];
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt)
        #pragma unroll
        for (int t = 0; t < KG; ++t) {
            const float* xp = X + (size_t)(rec[rt] < 0 ? 0 : rec[rt]) * IN + O::kidx(t, g, 0);
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
            if (rec[rt] >= 0) {
                if (O::steps(t) == 4) {
                    v = *(const SSLA_GLOBAL f32x4*)xp;
                } else {
                    v[0] = gload(xp);
                    v[1] = gload(xp + 1);
                }
            }
            xr[rt][t] = v;
        }
    f32x4 acc[RT][NT];
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt)
        #pragma unroll
        for (int ot = 0; ot < NT; ++ot) acc[rt][ot] = f32x4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();

    const SSLA_GLOBAL f32x4* wq = (const SSLA_GLOBAL f32x4*)po + lane;
    const SSLA_GLOBAL f32x4* wg = (const SSLA_GLOBAL f32x4*)(po + O::Q) + lane;
    // item it = delta * NT + ct: its q and goW fragments and the h values (an
    // absent pair, p < 0, reads row 0 and is zeroed where it is used, so the
    // loads carry no branch and the next item's stay in flight)
    auto load = [&](int it, f32x4 (&aq)[KG], f32x4 (&ag)[NT], f32x4 (&hv)[RT], int (&pv)[RT]) {
        const int d = it / NT, ct = it - d * NT;
        #pragma unroll
        for (int t = 0; t < KG; ++t) {
            const SSLA_GLOBAL f32x4* src = wq + ((size_t)it * KG + t) * 64;
            if (O::steps(t) == 4) {
                aq[t] = *src;
            } else {
                // a half group: the two live values only (a 16-byte load
                // would keep two dead registers in flight)
                const f32x2 v = *(const SSLA_GLOBAL f32x2*)src;
                aq[t] = f32x4{v[0], v[1], 0.f, 0.f};
            }
        }
        #pragma unroll
        for (int ot = 0; ot < NT; ++ot) ag[ot] = wg[((size_t)it * NT + ot) * 64];
        #pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int p = sp[16 * rt + j][d];
            pv[rt] = p;
            hv[rt] = *(const SSLA_GLOBAL f32x4*)(HR + (size_t)(p < 0 ? 0 : p) * OUT + 16 * ct + 4 * g);
        }
    };
    auto compute = [&](const f32x4 (&aq)[KG], const f32x4 (&ag)[NT], const f32x4 (&hv)[RT],
                       const int (&pv)[RT]) {
        f32x4 q[RT];
        #pragma unroll
        for (int rt = 0; rt < RT; ++rt) q[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
        #pragma unroll
        for (int t = 0; t < KG; ++t)
            #pragma unroll
            for (int i = 0; i < O::steps(t); ++i)
                #pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    q[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(aq[t][i], xr[rt][t][i], q[rt],
                                                                 0, 0, 0);
        #pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            q[rt] = pv[rt] >= 0 ? q[rt] * hv[rt] : f32x4{0.f, 0.f, 0.f, 0.f};
        #pragma unroll
        for (int i = 0; i < 4; ++i)
            #pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                #pragma unroll
                for (int ot = 0; ot < NT; ++ot)
                    acc[rt][ot] = __builtin_amdgcn_mfma_f32_16x16x4f32(ag[ot][i], q[rt][i],
                                                                       acc[rt][ot], 0, 0, 0);
    };
    // this wave's items: deltas [wv * 9 / KS, (wv + 1) * 9 / KS), the K parts
    // split over the KS waves.  The loop is unrolled (a fixed trip count, no
    // branches), and the scheduling barriers keep item k + 1's loads ahead of
    // item k's MFMAs: the wait before item k then covers only its own loads,
    // issued one item earlier.
    static_assert(kPatch % KS == 0, "K parts of whole deltas");
    constexpr int NI = kPatch / KS * NT;
    const int i0 = wv * NI;
    f32x4 aqb[2][KG], agb[2][NT], hvb[2][RT];
    int pvb[2][RT];
    load(i0, aqb[0], agb[0], hvb[0], pvb[0]);
    #pragma unroll
    for (int k = 0; k < NI; ++k) {
        if (k + 1 < NI)
            load(i0 + k + 1, aqb[(k + 1) & 1], agb[(k + 1) & 1], hvb[(k + 1) & 1], pvb[(k + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        compute(aqb[k & 1], agb[k & 1], hvb[k & 1], pvb[k & 1]);
        if constexpr (KS == 1) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (KS > 1) {
        if (wv > 0) {
            #pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                #pragma unroll
                for (int ot = 0; ot < NT; ++ot) part[wv - 1][rt * NT + ot][lane] = acc[rt][ot];
        }
        __syncthreads();
        if (wv > 0) return;
        #pragma unroll
        for (int w = 0; w < KS - 1; ++w)
            #pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                #pragma unroll
                for (int ot = 0; ot < NT; ++ot) acc[rt][ot] += part[w][rt * NT + ot][lane];
    }
    if constexpr (O::IP) {
        const SSLA_GLOBAL f32x4* wi = (const SSLA_GLOBAL f32x4*)(po + O::Q + O::GO) + lane;
        #pragma unroll
        for (int ot = 0; ot < NT; ++ot) {
            f32x4 ai[KG];
            #pragma unroll
            for (int t = 0; t < KG; ++t) ai[t] = wi[((size_t)ot * KG + t) * 64];
            #pragma unroll
            for (int t = 0; t < KG; ++t)
                #pragma unroll
                for (int i = 0; i < O::steps(t); ++i)
                    #pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                        acc[rt][ot] = __builtin_amdgcn_mfma_f32_16x16x4f32(ai[t][i], xr[rt][t][i],
                                                                           acc[rt][ot], 0, 0, 0);
        }
    } else {
        // residual: the lane holds X[rec][16 ot + 4 g + i] as xr[rt][ot][i]
        #pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            #pragma unroll
            for (int ot = 0; ot < NT; ++ot) acc[rt][ot] += xr[rt][ot];
    }
    // fp64 LayerNorm (eps 1e-5): lane (g, j) holds outputs 16 ot + 4 g + i of
    // record j of each tile; the record's sums are over lanes j + 16 g
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        double s = 0.0;
        #pragma unroll
        for (int ot = 0; ot < NT; ++ot)
            #pragma unroll
            for (int i = 0; i < 4; ++i) s += (double)acc[rt][ot][i];
        const double mean = sum4_lanes(s, lane) / (double)OUT;
        double v = 0.0;
        #pragma unroll
        for (int ot = 0; ot < NT; ++ot)
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double dd = (double)acc[rt][ot][i] - mean;
                v += dd * dd;
            }
        const double inv = 1.0 / sqrt(sum4_lanes(v, lane) / (double)OUT + 1e-5);
        #pragma unroll
        for (int ot = 0; ot < NT && rec[rt] >= 0; ++ot) {
            const int c = 16 * ot + 4 * g;
            const f32x4 ga = *(const SSLA_GLOBAL f32x4*)(gamma + c);
            const f32x4 be = *(const SSLA_GLOBAL f32x4*)(beta + c);
            f32x4 o;
            #pragma unroll
            for (int i = 0; i < 4; ++i)
                o[i] = (float)(((double)acc[rt][ot][i] - mean) * inv * (double)ga[i] +
                               (double)be[i]);
            *(SSLA_GLOBAL f32x4*)(Y + (size_t)rec[rt] * OUT + c) = o;
        }
    }
}

// The sum over each quad of lanes, in every lane of it: DPP quad_perm moves
// (xor 1, then xor 2) instead of LDS-permute shuffles.
__device__ __forceinline__ float quad_sum(float v) {
    v += __builtin_bit_cast(
        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
    v += __builtin_bit_cast(
        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false));
    return v;
}

// The prediction grid: a record's raw head row is published when it is the
// last owned pass-3 record of its s3 cell (k_tdrop3), with the number of such
// records added to the cell's version.  Each head kernel does it for the rows it
// has just computed (a launch of its own for it cost the small drains 8 us).
struct PredGrid {
    const unsigned char* owner;
    const uint32_t* key3_by_g;
    const int *last, *count;
    const BlockDesc* bd;
    Geometry G;
};

__device__ __forceinline__ void pred_write(const PredGrid& p, int g, const float* v7) {
    if (!p.owner[g]) return;
    const uint32_t k = p.key3_by_g[g];
    if (p.last[k] != g) return;
    const int b = (int)k / p.G.C3, cell = (int)k % p.G.C3;
    const HybridStrip& s = p.bd[b].strip;
    const int sx = cell % p.G.W3, sy = cell / p.G.W3;
    const int hx = sx - s.s3_owned_lo, hy = sy - s.s3_owned_y_lo;
    const int w = s.s3_owned_hi - s.s3_owned_lo, h = s.s3_owned_y_hi - s.s3_owned_y_lo;
    if (hx < 0 || hx >= w || hy < 0 || hy >= h) return;
    const int idx = hy * w + hx;
    publish_pred(p.bd[b].preds ? p.bd[b].preds + (size_t)idx * 7 : nullptr,
                 p.bd[b].version ? p.bd[b].version + idx : nullptr, v7, (unsigned)p.count[k]);
}

// ---------------------------------------------------------------------------
// head: raw [reg0..3, obj, cls0, cls1] for pass-3 records
// (...celled.cuh:841-902).  One workgroup = 64 records (list order): their
// 96-channel features staged in LDS; the two 1x1 convolutions (cls, reg; BN
// folded) as one 64 x 192 x 96 product of 16 x 16 MFMA tiles whose B
// operands are read straight from the row-major (IN, OUT) weights (lane l
// takes row 4s + l/16, column l%16 of step s); SiLU into LDS; then the
// seven prediction dot products, four threads per record.
// ---------------------------------------------------------------------------
constexpr int kHeadThreads = 64 * 2 * SSLA_C3 / kMT;      // a wave per column tile
__global__ void __launch_bounds__(kHeadThreads)
k_head(const int* __restrict__ n_dev, const int* __restrict__ list,
       const float* __restrict__ X, HeadPtrs hp, PredGrid pg, float* __restrict__ H7) {
    constexpr int C = SSLA_C3, XST = lds_stride(C), HST = 2 * C + 4, CT = 2 * C / kMT;
    __shared__ __align__(16) float xs[kTM * XST];
    __shared__ float hs[kTM * HST];           // [yc | yr] per record
    __shared__ int rows[kTM];
    const int n = *n_dev;
    const int base = blockIdx.x * kTM;
    if (base >= n) return;
    const int cnt = min(kTM, n - base);
    const int tid = threadIdx.x;
    if (tid < kTM) rows[tid] = tid < cnt ? list[base + tid] : -1;
    __syncthreads();
    constexpr int C4 = C / 4;
    for (int t = tid; t < kTM * C4; t += kHeadThreads) {
        const int r = t / C4, q = t - r * C4;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (rows[r] >= 0) v = reinterpret_cast<const float4*>(X)[(size_t)rows[r] * C4 + q];
        lds_put4(&xs[r * XST + 4 * q], v);
    }
    __syncthreads();
    const int lane = tid & 63, wv = tid >> 6, li = lane & 15, lk = lane >> 4;
    const int mtiles = (cnt + kMT - 1) / kMT;
    // column tiles 0..5: cls conv, 6..11: reg conv, one per wave
    {
        const int ct = wv;
        static_assert(kHeadThreads == 64 * CT, "a wave per column tile");
        const bool reg = ct >= CT / 2;
        const float* W = reg ? hp.reg_conv_W : hp.cls_conv_W;
        const float* bias = reg ? hp.reg_conv_b : hp.cls_conv_b;
        const int col = (reg ? ct - CT / 2 : ct) * kMT + li;
        float b[C / 4];
        #pragma unroll
        for (int s = 0; s < C / 4; ++s) b[s] = gload(W + (size_t)(4 * s + lk) * C + col);
        const float bc = bias[col];
        for (int m = 0; m < mtiles; ++m) {
            const float* a = &xs[(m * kMT + li) * XST + lk];
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            #pragma unroll
            for (int s = 0; s < C / 4; ++s)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[4 * s], b[s], acc, 0, 0, 0);
            #pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float y = acc[r] + bc;
                hs[(m * kMT + 4 * lk + r) * HST + ct * kMT + li] = y * sigmoid_fast(y);
            }
        }
    }
    __syncthreads();
    // predictions: record r = tid / 4, channels part, part + 4, ... (24 each)
    if (tid >= 4 * kTM) return;
    const int r = tid >> 2, part = tid & 3;
    float o[7];
    #pragma unroll
    for (int k = 0; k < 7; ++k) o[k] = 0.f;
    if (r < cnt) {
        const float* yc = &hs[r * HST];
        const float* yr = yc + C;
        // (unrolled: a rolled loop waits for one channel's seven weights at a time)
        #pragma unroll 6
        for (int i = part; i < C; i += 4) {
            #pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = fmaf(hp.reg_pred_W[(size_t)i * 4 + k], yr[i], o[k]);
            o[4] = fmaf(hp.obj_pred_W[i], yr[i], o[4]);
            #pragma unroll
            for (int k = 0; k < 2; ++k) o[5 + k] = fmaf(hp.cls_pred_W[(size_t)i * 2 + k], yc[i], o[5 + k]);
        }
    }
    #pragma unroll
    for (int k = 0; k < 7; ++k) o[k] = quad_sum(o[k]);
    if (r < cnt && part == 0) {
        float* out = H7 + (size_t)rows[r] * 7;
        #pragma unroll
        for (int k = 0; k < 4; ++k) o[k] += hp.reg_pred_b[k];
        o[4] += hp.obj_pred_b[0];
        o[5] += hp.cls_pred_b[0];
        o[6] += hp.cls_pred_b[1];
        #pragma unroll
        for (int k = 0; k < 7; ++k) out[k] = o[k];
        pred_write(pg, rows[r], o);
    }
}

// Single-linear head (...celled.cuh:1476-1481, matvec_w<C3, 7> over
// head_W (C3, 7) row-major, plus head_b) for pass-3 records: 64 records per
// workgroup in list order, four threads per record (channels part, part + 4,
// ...), the quad's partial sums added with two DPP moves.
__global__ void __launch_bounds__(256)
k_head_linear(const int* __restrict__ n_dev, const int* __restrict__ list,
              const float* __restrict__ X, HeadPtrs hp, PredGrid pg, float* __restrict__ H7) {
    constexpr int C = SSLA_C3;
    const int n = *n_dev;
    const int base = blockIdx.x * kTM;
    if (base >= n) return;
    const int j = base + (threadIdx.x >> 2), part = threadIdx.x & 3;
    const bool on = j < n;
    const int g = on ? list[j] : 0;
    float o[7];
    #pragma unroll
    for (int k = 0; k < 7; ++k) o[k] = 0.f;
    if (on) {
        const float* x = X + (size_t)g * C;
        for (int i = part; i < C; i += 4) {
            const float xi = x[i];
            #pragma unroll
            for (int k = 0; k < 7; ++k) o[k] = fmaf(hp.lin_W[(size_t)i * 7 + k], xi, o[k]);
        }
    }
    #pragma unroll
    for (int k = 0; k < 7; ++k) o[k] = quad_sum(o[k]);
    if (on && part == 0) {
        float* out = H7 + (size_t)g * 7;
        #pragma unroll
        for (int k = 0; k < 7; ++k) {
            o[k] += hp.lin_b[k];
            out[k] = o[k];
        }
        pred_write(pg, g, o);
    }
}

// Output slots (...celled.cuh:1233-1247 conventions) and raw head rows.
// Output slots (392 B = 49 eight-byte words) and head rows as coalesced
// 8-byte stores: 128 records per 256-thread workgroup (a small call: 8, so that
// its few records are not one workgroup's loop).
constexpr int kEmitRec = 128, kEmitRecFew = 8;

template <int RPB>
__global__ void __launch_bounds__(256)
k_emit(int E, const BlockDesc* __restrict__ bd, int nb,
       const int* __restrict__ cell2,
       const unsigned char* __restrict__ owner,
       const unsigned char* __restrict__ pass2,
       const unsigned char* __restrict__ pass3,
       const float* __restrict__ X4, const float* __restrict__ H7,
       int have_head) {
    constexpr int NW = (int)(sizeof(HybridS2S3OutputSlot) / 8);
    static_assert(sizeof(HybridS2S3OutputSlot) % 8 == 0 && SSLA_C3 % 2 == 0, "slot words");
    __shared__ int sb[RPB], sk[RPB], sp2[RPB], sp3[RPB];
    __shared__ unsigned char sfeat[RPB], shead[RPB];
    const int g0 = blockIdx.x * RPB;
    const int t = threadIdx.x;
    if (t < RPB) {
        const int g = g0 + t;
        int b = 0, k = -1, q2 = -2, q3 = -2;
        bool feat = false, head = false;
        if (g < E) {
            b = find_block(bd, nb, g);
            k = g - bd[b].offset;
            const bool valid = cell2[g] >= 0;
            const bool p2 = valid && pass2[g], p3 = p2 && pass3[g], own = owner[g];
            if (valid) {
                q2 = own ? (p2 ? 1 : 0) : -1;
                q3 = own ? (p3 ? 1 : 0) : -1;
            }
            feat = p3;
            head = have_head && p3 && own;
        }
        sb[t] = b; sk[t] = k; sp2[t] = q2; sp3[t] = q3;
        sfeat[t] = feat; shead[t] = head;
    }
    __syncthreads();
    for (int j = t; j < RPB * NW; j += 256) {
        const int r = j / NW, w = j - r * NW;
        const int k = sk[r];
        HybridS2S3OutputSlot* out = k >= 0 ? bd[sb[r]].out : nullptr;
        if (!out) continue;
        if (w == 0) {
            reinterpret_cast<int2*>(out + k)[0] = make_int2(sp2[r], sp3[r]);
        } else {
            const int i = 2 * (w - 1);
            float2 f = make_float2(0.f, 0.f);
            if (sfeat[r]) f = *reinterpret_cast<const float2*>(X4 + (size_t)(g0 + r) * SSLA_C3 + i);
            reinterpret_cast<float2*>(out[k].s3_feat)[w - 1] = f;
        }
    }
    for (int j = t; j < RPB * 7; j += 256) {
        const int r = j / 7, c = j - r * 7;
        const int k = sk[r];
        float* ho = k >= 0 ? bd[sb[r]].head_out : nullptr;
        if (ho) ho[(size_t)k * 7 + c] = shead[r] ? H7[(size_t)(g0 + r) * 7 + c] : 0.f;
    }
}

// ---------------------------------------------------------------------------
// workspace
// ---------------------------------------------------------------------------
struct Workspace {
    int cap = 0;            // records
    int cap_blocks = 0;
    int cap_keys = 0;
    void* base = nullptr;
    size_t bytes = 0;
    float *X0, *X1, *X2, *X3, *X4, *HR, *H7;   // HR: h rows of one layer, row 9 record + delta
    int *cell2, *list2, *list3, *counts;
    int *st2, *en2, *st3, *en3, *pst2, *pst3, *pcnt, *last3, *cnt3;
    uint2 *pent2, *pent3;                      // per sorted pair: {9 record + delta | need, cell key}
    int *goff2, *goff3;                        // first published-word slot of every key
    int *sidx;                                 // sorted s2 position of every record
    int *n2, *t3, *n3;                         // pass-2 records per s2 / s3 key, pass-3 per s3 key
    int *off2, *off3;                          // first pass-2 / pass-3 list slot of every key
    int *bh;                                   // radix-sort tile histograms
    unsigned char* old2;                       // s2 counters before the call
    unsigned long long* sw;                    // k_pscan: published words, per group
    int *ghist, *gw, *gcnt, *gend, *gstart, *gbase;          // s2 group order tables
    int4* glist;                                             // group of every s2 ticket
    int *ghist3, *gw3, *gcnt3, *gend3, *gstart3, *gbase3;    // ... and of the s3 level
    int4* glist3;
    int* scan_err = nullptr;                   // host memory: a look-back wait ran out
    unsigned char *owner, *pass2, *pass3;
    uint32_t *ka, *kb, *va, *vb, *key3g;
    BlockDesc* bd;
    hipEvent_t done = nullptr;         // the last drain's work on the workspace
    hipStream_t side = nullptr;        // s3 ordering, concurrent with L4 and L5
    hipEvent_t s2_ordered = nullptr;   // s2 tables and pass2 are complete
    hipEvent_t s3_ordered = nullptr;   // s3 tables and pass3 are complete
    hipEvent_t side_done = nullptr;    // the side stream's last work of a call
    int bh_ints = 0;
    int cus = 0;                       // compute units of the device
    int clk_khz = 0;                   // wall-clock (s_memrealtime) rate
    float* packed = nullptr;           // fragment-order weight copies (packed_weight_floats_d)
    PackedWeights pk = {};
    // phase timings of calls made without sync: their events, read and added
    // to the caller's array when a later call with sync returns
    struct Pending {
        hipEvent_t ev[SSLA_DRAIN_PHASES + 1];
        float* phase_ms;
        unsigned long long pmask;
    };
    std::vector<Pending> pending;
};
constexpr size_t kMaxPending = 256;    // more waiting calls: the oldest is waited for

// Adds the phase times of the oldest `n` pending calls to their arrays and
// frees their events (waiting for each event first).
int flush_pending(Workspace& w, size_t n) {
    n = std::min(n, w.pending.size());
    int rc = SSLA_OK;
    for (size_t i = 0; i < n; ++i) {
        Workspace::Pending& p = w.pending[i];
        for (int k = 0; k < SSLA_DRAIN_PHASES && rc == SSLA_OK; ++k) {
            if (!((p.pmask >> k) & 1ull) || !p.ev[k] || !p.ev[k + 1]) continue;
            float ms = 0.f;
            hipError_t e = hipEventSynchronize(p.ev[k + 1]);
            if (e == hipSuccess) e = hipEventElapsedTime(&ms, p.ev[k], p.ev[k + 1]);
            if (e != hipSuccess) {
                set_error(std::string("drain phase timing: ") + hipGetErrorString(e));
                rc = SSLA_ERR_HIP;
                break;
            }
            p.phase_ms[k] += ms;
        }
        for (int k = 0; k <= SSLA_DRAIN_PHASES; ++k)
            if (p.ev[k]) (void)hipEventDestroy(p.ev[k]);
    }
    w.pending.erase(w.pending.begin(), w.pending.begin() + n);
    return rc;
}

std::mutex g_ws_mu;
Workspace g_ws;
unsigned g_scan_tag = 0;     // tag of k_pscan's last launch (under g_ws_mu)

#define HIPCHK(call)                                                          \
    do {                                                                      \
        hipError_t e_ = (call);                                               \
        if (e_ != hipSuccess) {                                               \
            set_error(std::string(#call) + ": " + hipGetErrorString(e_));    \
            return SSLA_ERR_HIP;                                              \
        }                                                                     \
    } while (0)

size_t align_up(size_t v) { return (v + 255) & ~size_t(255); }

int ensure_workspace(int E, int nkeys) {
    if (E <= g_ws.cap && nkeys <= g_ws.cap_keys) return SSLA_OK;
    if (g_ws.base) {
        // the last drain's kernels (both streams, joined into `done`) are the
        // only users of the old workspace
        HIPCHK(hipEventSynchronize(g_ws.done));
        HIPCHK(hipFree(g_ws.base));
        g_ws.base = nullptr;
        g_ws.cap = 0;
    }
    const int cap = std::max(E, std::max(g_ws.cap, 1024));
    const int ck = std::max(nkeys, g_ws.cap_keys);
    const size_t P = (size_t)cap * kPatch;
    // group bound: full groups + one tail per key (shared groups are fewer
    // than the keys in them)
    const size_t mg = P / kGP + (size_t)ck + 1;
    // a cell's pairs come from distinct records: at most cap, so a cell has at
    // most cap / kGP + 1 groups
    const size_t nv = (size_t)cap / kGP + 3;
    // radix-sort tile histograms: (1 << kRMaxBits) digits x tiles
    const size_t bh = ((size_t)1 << kRMaxBits) * (size_t)((cap + kRTile - 1) / kRTile);
    struct Item { void** dst; size_t bytes; };
    Workspace& w = g_ws;
    std::vector<Item> items = {
        {(void**)&w.X0, sizeof(float) * (size_t)cap * SSLA_C1},
        {(void**)&w.X1, sizeof(float) * (size_t)cap * SSLA_C2},
        {(void**)&w.X2, sizeof(float) * (size_t)cap * SSLA_C2},
        {(void**)&w.X3, sizeof(float) * (size_t)cap * SSLA_C3},
        {(void**)&w.X4, sizeof(float) * (size_t)cap * SSLA_C3},
        {(void**)&w.HR, sizeof(float) * P * SSLA_C3},
        {(void**)&w.H7, sizeof(float) * (size_t)cap * 7},
        {(void**)&w.cell2, sizeof(int) * (size_t)cap},
        {(void**)&w.pent2, sizeof(uint2) * P},
        {(void**)&w.pent3, sizeof(uint2) * P},
        {(void**)&w.list2, sizeof(int) * (size_t)cap},
        {(void**)&w.list3, sizeof(int) * (size_t)cap},
        {(void**)&w.counts, sizeof(int) * 16},
        {(void**)&w.st2, sizeof(int) * (size_t)ck},
        {(void**)&w.en2, sizeof(int) * (size_t)ck},
        {(void**)&w.st3, sizeof(int) * (size_t)ck},
        {(void**)&w.en3, sizeof(int) * (size_t)ck},
        {(void**)&w.pst2, sizeof(int) * (size_t)ck},
        {(void**)&w.pst3, sizeof(int) * (size_t)ck},
        {(void**)&w.pcnt, sizeof(int) * (size_t)ck},
        {(void**)&w.last3, sizeof(int) * (size_t)ck},
        {(void**)&w.cnt3, sizeof(int) * (size_t)ck},
        {(void**)&w.owner, (size_t)cap},
        {(void**)&w.pass2, (size_t)cap},
        {(void**)&w.pass3, (size_t)cap},
        {(void**)&w.ka, sizeof(uint32_t) * (size_t)cap},
        {(void**)&w.kb, sizeof(uint32_t) * (size_t)cap},
        {(void**)&w.va, sizeof(uint32_t) * (size_t)cap},
        {(void**)&w.vb, sizeof(uint32_t) * (size_t)cap},
        {(void**)&w.key3g, sizeof(uint32_t) * (size_t)cap},
        {(void**)&w.sidx, sizeof(int) * (size_t)cap},
        {(void**)&w.goff2, sizeof(int) * (size_t)ck},
        {(void**)&w.goff3, sizeof(int) * (size_t)ck},
        {(void**)&w.n2, sizeof(int) * (size_t)ck},
        {(void**)&w.t3, sizeof(int) * (size_t)ck},
        {(void**)&w.n3, sizeof(int) * (size_t)ck},
        {(void**)&w.off2, sizeof(int) * (size_t)ck},
        {(void**)&w.off3, sizeof(int) * (size_t)ck},
        {(void**)&w.bh, sizeof(int) * bh},
        {(void**)&w.old2, (size_t)ck},
        {(void**)&w.sw, sizeof(unsigned long long) * mg * 3 * SSLA_C3},
        {(void**)&w.ghist, sizeof(int) * nv},
        {(void**)&w.gstart, sizeof(int) * nv},
        {(void**)&w.gbase, sizeof(int) * nv},
        {(void**)&w.gw, sizeof(int) * (size_t)ck},
        {(void**)&w.gcnt, sizeof(int) * (size_t)ck},
        {(void**)&w.gend, sizeof(int) * (size_t)ck},
        {(void**)&w.glist, sizeof(int4) * mg},
        {(void**)&w.ghist3, sizeof(int) * nv},
        {(void**)&w.gstart3, sizeof(int) * nv},
        {(void**)&w.gbase3, sizeof(int) * nv},
        {(void**)&w.gw3, sizeof(int) * (size_t)ck},
        {(void**)&w.gcnt3, sizeof(int) * (size_t)ck},
        {(void**)&w.gend3, sizeof(int) * (size_t)ck},
        {(void**)&w.glist3, sizeof(int4) * mg},
        {(void**)&w.bd, sizeof(BlockDesc) * SSLA_MAX_BLOCKS},
    };
    size_t total = 0;
    for (auto& it : items) total += align_up(it.bytes);
    void* base = nullptr;
    HIPCHK(hipMalloc(&base, total));
    char* p = static_cast<char*>(base);
    for (auto& it : items) {
        *it.dst = p;
        p += align_up(it.bytes);
    }
    // no stale word may carry a future launch's tag
    HIPCHK(hipMemset(w.sw, 0, sizeof(unsigned long long) * mg * 3 * SSLA_C3));
    if (!w.scan_err) {
        HIPCHK(hipHostMalloc((void**)&w.scan_err, sizeof(int), hipHostMallocCoherent));
        *w.scan_err = 0;
    }
    if (!w.done) {
        HIPCHK(hipEventCreateWithFlags(&w.done, hipEventDisableTiming));
        HIPCHK(hipEventCreateWithFlags(&w.s2_ordered, hipEventDisableTiming));
        HIPCHK(hipEventCreateWithFlags(&w.s3_ordered, hipEventDisableTiming));
        HIPCHK(hipEventCreateWithFlags(&w.side_done, hipEventDisableTiming));
        HIPCHK(hipStreamCreateWithFlags(&w.side, hipStreamNonBlocking));
        HIPCHK(hipMalloc(&w.packed, sizeof(float) * packed_weight_floats_d()));
        int dev = 0;
        HIPCHK(hipGetDevice(&dev));
        HIPCHK(hipDeviceGetAttribute(&w.cus, hipDeviceAttributeMultiprocessorCount, dev));
        HIPCHK(hipDeviceGetAttribute(&w.clk_khz, hipDeviceAttributeWallClockRate, dev));
    }
    w.base = base;
    w.bytes = total;
    w.cap = cap;
    w.cap_keys = ck;
    w.bh_ints = (int)bh;
    return SSLA_OK;
}

int bits_for(uint32_t v) {
    int b = 1;
    while ((1u << b) <= v && b < 32) ++b;
    return b;
}

inline unsigned grid1(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// Every return of a call after its first launch passes through finish():
// the side stream's work joins `st`, and `done` marks the end of the call's
// use of the workspace, so the next call (on any stream) and a workspace
// regrowth wait for all of it -- also when the call stops at an error.
struct CallEnd {
    Workspace& w;
    hipStream_t st;
    bool side = false;         // the call has launched on the side stream
    bool ended = false;
    void finish() {
        if (ended) return;
        ended = true;
        if (side) {
            (void)hipEventRecord(w.side_done, w.side);
            (void)hipStreamWaitEvent(st, w.side_done, 0);
        }
        (void)hipEventRecord(w.done, st);
    }
    ~CallEnd() { finish(); }
};

}  // namespace

namespace {
// zero fill of n bytes at p (16-byte stores for the aligned body)
__global__ void k_zero_bytes(unsigned char* __restrict__ p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t n16 = n >> 4;
    if (i < n16) reinterpret_cast<uint4*>(p)[i] = make_uint4(0u, 0u, 0u, 0u);
    if (i < (n & 15)) p[(n16 << 4) + i] = 0;
}
}  // namespace

int zero_async(void* p, size_t nbytes, hipStream_t st) {
    if (!nbytes) return SSLA_OK;
    if (!p || (reinterpret_cast<uintptr_t>(p) & 15)) {
        set_error("zero_async: null or unaligned pointer");
        return SSLA_ERR_ARG;
    }
    const size_t n16 = std::max<size_t>(nbytes >> 4, 16);
    hipLaunchKernelGGL(k_zero_bytes, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, st,
                       static_cast<unsigned char*>(p), nbytes);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string("zero_async: ") + hipGetErrorString(e));
        return SSLA_ERR_HIP;
    }
    return SSLA_OK;
}

int drain_reserve(const HybridS2S3Config* cfg, int max_records) {
    if (!cfg || cfg->n_blocks < 1 || cfg->n_blocks > SSLA_MAX_BLOCKS || cfg->H2 <= 0 ||
        cfg->W2 <= 0 || cfg->H2 > 65535 || cfg->W2 > 65535 || max_records < 0 ||
        (long long)max_records * kPatch > 0x7fffffffLL ||
        (long long)cfg->n_blocks * cfg->H2 * cfg->W2 >= 0x7fffffffLL) {
        set_error("drain_reserve: bad configuration or record count");
        return SSLA_ERR_ARG;
    }
    std::lock_guard<std::mutex> lock(g_ws_mu);
    return ensure_workspace(std::max(max_records, 1), cfg->n_blocks * cfg->H2 * cfg->W2 + 1);
}

int scan_drain(const HybridS2S3Config* cfg, const HybridInputRec* const* rings,
               const int* ns, HybridS2S3OutputSlot* const* outs,
               float* const* head_outs, hipStream_t st, bool sync,
               float* phase_ms, unsigned long long phase_mask) {
    const int nb = cfg->n_blocks;
    if (nb < 1 || nb > SSLA_MAX_BLOCKS) {
        set_error("n_blocks must be in [1, 16]");
        return SSLA_ERR_ARG;
    }
    if (cfg->H2 <= 0 || cfg->W2 <= 0 || (cfg->H2 & 1) || (cfg->W2 & 1) ||
        cfg->H3 != cfg->H2 / 2 || cfg->W3 != cfg->W2 / 2 ||
        cfg->H2 > 65535 || cfg->W2 > 65535) {
        set_error("grid must have even H2, W2 and H3 = H2/2, W3 = W2/2");
        return SSLA_ERR_ARG;
    }
    for (int b = 0; b < nb; ++b) {
        for (int li = 0; li < 4; ++li) {
            const LayerWeightsS2S3& L = cfg->layers[b][li];
            const LayerWeightsS2S3& L0 = cfg->layers[0][li];
            if (!L.qvgIn || !L.goW || !L.ln_gamma || !L.ln_beta) {
                set_error("layer weights not bound for block " + std::to_string(b));
                return SSLA_ERR_ARG;
            }
            if (L.qvgIn != L0.qvgIn || L.goW != L0.goW || L.input_proj != L0.input_proj ||
                L.ln_gamma != L0.ln_gamma || L.ln_beta != L0.ln_beta) {
                set_error("all blocks must share one set of layer weights");
                return SSLA_ERR_ARG;
            }
            if (!cfg->hidden[b][li]) {
                set_error("hidden state not allocated for block " + std::to_string(b));
                return SSLA_ERR_ARG;
            }
        }
        if (!cfg->tdrop_s2[b] || !cfg->tdrop_s3[b]) {
            set_error("tdrop counters not allocated for block " + std::to_string(b));
            return SSLA_ERR_ARG;
        }
        if (ns[b] < 0 || (ns[b] > 0 && !rings[b])) {
            set_error("bad ring / count for block " + std::to_string(b));
            return SSLA_ERR_ARG;
        }
    }
    if ((cfg->layers[0][0].input_proj == nullptr) || (cfg->layers[0][2].input_proj == nullptr) ||
        cfg->layers[0][1].input_proj != nullptr || cfg->layers[0][3].input_proj != nullptr) {
        set_error("L4/L6 need input_proj and L5/L7 must not have one");
        return SSLA_ERR_ARG;
    }
    long long E64 = 0;
    for (int b = 0; b < nb; ++b) E64 += ns[b];
    if (E64 * kPatch > 0x7fffffffLL) {
        set_error("too many records in one call");
        return SSLA_ERR_ARG;
    }
    const int E = (int)E64;
    Geometry G;
    G.H2 = cfg->H2; G.W2 = cfg->W2; G.H3 = cfg->H3; G.W3 = cfg->W3;
    G.C2 = G.H2 * G.W2; G.C3 = G.H3 * G.W3; G.nb = nb; G.window = cfg->tdrop_window;
    const uint32_t nk2 = (uint32_t)(nb * G.C2), nk3 = (uint32_t)(nb * G.C3);
    const int head = head_kind(cfg);
    const bool have_head = head != kHeadNone;
    if (const char* m = head_missing(cfg)) {
        set_error(m);
        return SSLA_ERR_ARG;
    }

    std::lock_guard<std::mutex> lock(g_ws_mu);
    if (E == 0) return SSLA_OK;
    {
        const int rc = ensure_workspace(E, (int)nk2 + 1);
        if (rc) return rc;
    }
    Workspace& w = g_ws;
    CallEnd end{w, st};

    BlockTable tab;
    std::memset(&tab, 0, sizeof tab);
    BlockDesc* hbd = tab.d;
    int off = 0;
    for (int b = 0; b < nb; ++b) {
        BlockDesc& d = hbd[b];
        d.ring = rings[b];
        d.out = outs ? outs[b] : nullptr;
        d.head_out = head_outs ? head_outs[b] : nullptr;
        for (int li = 0; li < 4; ++li) d.hidden[li] = cfg->hidden[b][li];
        d.td2 = cfg->tdrop_s2[b];
        d.td3 = cfg->tdrop_s3[b];
        d.preds = have_head ? cfg->preds[b] : nullptr;
        d.version = have_head ? cfg->version[b] : nullptr;
        d.strip = cfg->strip[b];
        d.n = ns[b];
        d.offset = off;
        off += ns[b];
    }
    // blocks with n == 0 must not capture records: move their offset past E.
    for (int b = 0; b < nb; ++b)
        if (hbd[b].n == 0) hbd[b].offset = E + 1;
    // Calls share one workspace: a call on another stream runs after the
    // previous call's kernels (device-side wait, the host does not block).
    HIPCHK(hipStreamWaitEvent(st, w.done, 0));

    // Phase timing (optional): events recorded on `st` at the boundaries of
    // the phases in pmask only -- each event costs a few microseconds of
    // queue time between the kernels it separates.
    hipEvent_t ev[SSLA_DRAIN_PHASES + 1] = {};
    int n_mark = 0;
    const unsigned long long pmask = phase_ms ? (phase_mask ? phase_mask : ~0ull) : 0ull;
    struct EvFree {
        hipEvent_t* ev;
        ~EvFree() {
            for (int k = 0; k <= SSLA_DRAIN_PHASES; ++k)
                if (ev[k]) (void)hipEventDestroy(ev[k]);
        }
    } ev_free{ev};
    auto mark = [&]() -> int {
        const int b = n_mark++;                       // boundary b opens phase b
        if (b > SSLA_DRAIN_PHASES) return SSLA_OK;
        if (!((pmask >> b) & 1ull) && !(b > 0 && ((pmask >> (b - 1)) & 1ull))) return SSLA_OK;
        HIPCHK(hipEventCreate(&ev[b]));
        HIPCHK(hipEventRecord(ev[b], st));
        return SSLA_OK;
    };
#define MARK() do { const int rc_ = mark(); if (rc_) return rc_; } while (0)
    // fragment-order copies of the layer weights for the MFMA kernels, rebuilt
    // by every call (in k_decode's launch), so weights rewritten in place by
    // any means are always the ones used
    const PackSrc psrc = pack_setup<true>(cfg->layers[0], w.packed, &w.pk);
    const PackedWeights& pk = w.pk;
    MARK();
    const LayerWeightsS2S3* L = cfg->layers[0];
    const bool small = E <= kSmallRec && nk2 <= (uint32_t)kScanThreads;
    const bool small_all = small && E <= kSmallAll;      // the s3 ordering too
    uint32_t *K2 = w.ka, *V2 = w.va, *K3 = w.kb, *V3 = w.vb;
    hipStream_t s3 = w.side;
    // per-call fills: run bounds of the s2 keys (k_runs writes those that
    // occur), the list and group counters, the prediction-grid writers
    // the group-count bound of this call's cells (see ensure_workspace), and
    // whether a level's group list fits the key scan's LDS
    const int nv = E / kGP + 3;
    const bool gt2 = nk2 <= (uint32_t)kScanThreads && nv <= kGroupLds;
    const bool gt3 = nk3 <= (uint32_t)kScanThreads && nv <= kGroupLds;
    FillSet f{};
    {
        int* arr[kFills] = {w.st2, w.en2, w.counts, w.last3, w.cnt3, w.ghist, w.ghist3};
        const int len[kFills] = {(int)nk2, (int)nk2, 16, have_head ? (int)nk3 : 0,
                                 have_head ? (int)nk3 : 0, gt2 ? 0 : nv, gt3 ? 0 : nv};
        const int val[kFills] = {0, 0, 0, -1, 0, 0, 0};
        for (int i = 0; i < kFills; ++i) {
            f.p[i] = arr[i];
            f.n[i] = len[i];
            f.v[i] = val[i];
        }
    }
    if (small) {
        const int npk = (int)((PackLayout<true>::off[8] + kScanThreads - 1) / kScanThreads);
        const SmallOut o{w.cell2, w.owner, w.pass2, w.pass3, w.list2, w.list3, w.counts, w.last3,
                         w.cnt3, w.key3g, w.pent2, w.pent3, w.glist, w.glist3, have_head ? 1 : 0,
                         K2, V2, w.sidx, w.st2, w.en2, w.pst2, w.n2, w.off2, w.old2};
        const dim3 grid(1 + npk + grid1(E, kScanThreads / 8));
        if (small_all)
            hipLaunchKernelGGL(k_small_order<true>, grid, dim3(kScanThreads), 0, st, E, tab, w.bd, G,
                               w.X0, o, psrc, w.packed, npk);
        else
            hipLaunchKernelGGL(k_small_order<false>, grid, dim3(kScanThreads), 0, st, E, tab, w.bd, G,
                               w.X0, o, psrc, w.packed, npk);
    } else {
        // ---- decode (and the fills); stable radix sort of the records by s2 key --
        {
            const int ndec = (int)grid1(E, kDecRec), fblk = (int)grid1(std::max<int>(std::max<int>((int)nk2, 16), nv), 256);
            const int npk = (int)((PackLayout<true>::off[8] + 255) / 256);
            hipLaunchKernelGGL(k_decode, dim3(ndec + fblk * kFills + npk + 1), dim3(256), 0, st, E, tab,
                               w.bd, G, w.X0, w.cell2, w.owner, w.ka, w.va, ndec, f, fblk, psrc,
                               w.packed, npk);
        }
        const int bits2 = bits_for(nk2);
        const int passes = (bits2 + kRMaxBits - 1) / kRMaxBits;
        const int T = (int)grid1(E, kRTile);
        uint32_t *kin = w.ka, *vin = nullptr, *kout = w.kb, *vout = w.vb;
        for (int ps = 0, shift = 0; ps < passes; ++ps) {
            const int bits = (bits2 - shift + (passes - ps) - 1) / (passes - ps);
            if ((1 << bits) * T > w.bh_ints) {
                set_error("drain: radix histogram larger than its workspace");
                return SSLA_ERR_STATE;
            }
            // a one-pass sort's digit is the whole key: bins for the keys present
            // (nk2 values and the keyless records' nk2) only
            const int nbins = passes == 1 ? (int)nk2 + 1 : 1 << bits;
            hipLaunchKernelGGL(k_rs_hist, dim3(T), dim3(kRThreads), 0, st, E, kin, shift, bits, nbins,
                               T, w.bh);
            hipLaunchKernelGGL(k_exscan, dim3(1), dim3(kScanThreads), 0, st, nbins * T, w.bh);
            hipLaunchKernelGGL(k_rs_scatter, dim3(T), dim3(kRThreads), 0, st, E, kin, vin, kout, vout,
                               ps == passes - 1 ? w.sidx : nullptr, shift, bits, nbins, T, w.bh);
            shift += bits;
            // the next pass writes the pair of buffers this pass read from
            uint32_t* const k2 = kout == w.kb ? w.ka : w.kb;
            uint32_t* const v2 = vout == w.vb ? w.va : w.vb;
            kin = kout;
            vin = vout;
            kout = k2;
            vout = v2;
        }
        // the sorted s2 order, and the buffers the s3 order is placed in
        K2 = kin;
        V2 = vin;
        K3 = kout;
        V3 = vout;
        // ---- counters, tdrop_s2, the pass-2 list, s2 pair and group tables -----
        if (passes == 1 && nk2 <= (uint32_t)kScanThreads) {
            // the one pass's histogram holds the run bounds: the key tables and
            // their scans in one workgroup
            const KeyHist kh{G.C2, G.W2, G.H2, T, G.window, (const int*)w.bh, w.st2, w.en2, w.bd,
                             w.old2};
            if (gt2)
                hipLaunchKernelGGL((k_keyscan<true, true>), dim3(1), dim3(kScanThreads), 0, st, (int)nk2,
                                   (const int*)nullptr, w.pst2, (int*)nullptr, w.goff2, w.n2, w.off2,
                                   w.counts + 0, kh, GroupTab{nv, w.glist, w.counts + 6});
            else
                hipLaunchKernelGGL((k_keyscan<true, false>), dim3(1), dim3(kScanThreads), 0, st, (int)nk2,
                                   (const int*)nullptr, w.pst2, (int*)nullptr, w.goff2, w.n2, w.off2,
                                   w.counts + 0, kh, GroupTab{});
        } else {
            hipLaunchKernelGGL(k_runs, dim3(grid1(E, 256)), dim3(256), 0, st, E, K2, nk2, w.st2, w.en2);
            hipLaunchKernelGGL(k_keys2, dim3(grid1(nk2, 256)), dim3(256), 0, st, nk2, G.C2, G.W2, G.H2,
                               w.st2, w.en2, w.bd, G.window, w.old2, w.n2, w.pcnt);
            if (gt2)
                hipLaunchKernelGGL((k_keyscan<false, true>), dim3(1), dim3(kScanThreads), 0, st, (int)nk2,
                                   w.pcnt, w.pst2, (int*)nullptr, w.goff2, w.n2, w.off2, w.counts + 0,
                                   KeyHist{}, GroupTab{nv, w.glist, w.counts + 6});
            else
                hipLaunchKernelGGL((k_keyscan<false, false>), dim3(1), dim3(kScanThreads), 0, st, (int)nk2,
                                   w.pcnt, w.pst2, (int*)nullptr, w.goff2, w.n2, w.off2, w.counts + 0,
                                   KeyHist{}, GroupTab{});
        }
    }
    if (!small_all) {
        const unsigned nbr = grid1(E, 256);
#define S2_TABLES(SMALL)                                                                              \
    hipLaunchKernelGGL(k_s2_tables<SMALL>, dim3(nbr + (gt2 ? 0u : grid1(nk2, 256))), dim3(256), 0, st, E, \
                       (int)nbr, K2, V2, nk2, G.C2, G.W2, G.H2, w.st2, w.en2, w.pst2, w.old2, w.off2,  \
                       G.window, w.pass2, w.list2, w.pent2, w.gcnt, w.gend, w.ghist, w.gw)
        if (E <= kSmallRec) S2_TABLES(true);
        else S2_TABLES(false);
#undef S2_TABLES
        if (!gt2)
            hipLaunchKernelGGL(k_group_order, dim3(1), dim3(kScanThreads), 0, st, (int)nk2, nv, w.pst2,
                               w.goff2, w.gcnt, w.gend, w.ghist, w.gw, w.gstart, w.gbase, w.glist,
                               w.counts + 6);
        // The s3 ordering needs only the s2 order, pass2 and the old counters, so
        // it runs on the side stream while L4 and L5 run here; L6 waits for it.
        // Its launches are sized by E; the pass-2 count stays on the device.  Its
        // event sits before L4's projection, so the side stream's small kernels
        // start beside the projection rather than beside the latency-bound parts
        // that follow it.
        HIPCHK(hipEventRecord(w.s2_ordered, st));
        end.side = true;
        HIPCHK(hipStreamWaitEvent(s3, w.s2_ordered, 0));
    }
    MARK();
    // The pass-2 and pass-3 counts stay on the device; the launches over their
    // lists are sized by bounds the host has.  A cell's L records in a row take
    // at most L P / 256 + 2 passes of the tdrop gate, P = ceil(256 / window)
    // the passing counter values per 256: any 256 consecutive values hold P,
    // and a shorter run, cut in two by the wrap, at most a1 / w + a2 / w + 2.
    const long long Pw = G.window <= 1 ? 256 : (256 + G.window - 1) / G.window;
    const int nmax2 = (int)std::min<long long>(E, ((long long)E * Pw + 255) / 256 + 2LL * nk2);
    const int nmax3 = (int)std::min<long long>(nmax2, ((long long)nmax2 * Pw + 255) / 256 + 2LL * nk3);
    const unsigned tiles3 = grid1(nmax3, kTM);
    const int* const no_count = nullptr;
    const int* const no_list = nullptr;
    // P + S of layer LI over the groups of level LV (their count in
    // counts[NG], ticket counter counts[8 + LI]): h rows to HR where the pair's
    // record needs the output (ALL: every pair's).  One workgroup of k_pscan
    // fits a CU (155,136 B of LDS, 1024 threads), and the grid is one per CU, or
    // the groups the call can have if they are fewer: full groups, a tail per cell
    // of more than kGW pairs and the shared ones, one per window of kGW.
    const unsigned long long wait_ticks = (unsigned long long)std::max(w.clk_khz, 1) * 500ull;
    const unsigned cus = w.cus > 0 ? (unsigned)w.cus : 256u;
    auto group_bound = [](long long recs, long long nk) {
        const long long p = recs * kPatch, small = p / kGW + 1;
        return p / kGP + 2 * std::min(nk, small);
    };
    auto ps_grid = [&](long long groups, int slabs) {
        return (unsigned)std::min<long long>(groups * slabs, cus);
    };
    const unsigned gridS4 = ps_grid(group_bound(E, nk2), 1);
    const unsigned gridS6 = ps_grid(group_bound(nmax2, nk3), SSLA_C3 / kPSC);
#define PSCAN(IN, OUT, NT, LI, LV, NG, GL, ALL, XIN, CELLS, GRID)                                    \
    do {                                                                                            \
        unsigned tag_ = ++g_scan_tag;                                                               \
        if (tag_ == 0) tag_ = ++g_scan_tag;                                                         \
        hipLaunchKernelGGL((k_pscan<IN, OUT, ALL, NT>), dim3(GRID), dim3(kPSThreads), 0, st,             \
                           (const int*)(w.counts + NG), w.counts + 8 + LI, tag_, GL, w.pent##LV,     \
                           XIN, pk.pp[LI], CELLS, w.bd, LI, w.HR, w.sw, w.scan_err, wait_ticks);    \
        MARK();                                                                                     \
        MARK();                                                                                     \
        MARK();                                                                                     \
        MARK();                                                                                     \
    } while (0)
    // ---- L4: 24 -> 48, all records ----------------------------------------
    PSCAN(SSLA_C1, SSLA_C2, true, 0, 2, 6, w.glist, true, w.X0, G.C2, gridS4);
    const auto few = [&](int n) { return grid1(n, 16) <= 2 * cus; };
#define OUTT(LI, IN, OUT, RT, KS, WPS, KSF, N, COUNT, LIST, XIN, SH, WL, HL, XOUT)                           \
    do {                                                                                            \
        if (few(N))                                                                                 \
            hipLaunchKernelGGL((k_outt<IN, OUT, 1, KSF>), dim3(grid1(N, 16)),                        \
                               dim3(64 * KSF), 0, st, E, COUNT, LIST, XIN, w.cell2, SH, G.W2,  \
                               WL, HL, w.HR, pk.po[LI], L[LI].ln_gamma, L[LI].ln_beta, XOUT);       \
        else                                                                                        \
            hipLaunchKernelGGL((k_outt<IN, OUT, RT, KS, WPS>), dim3(grid1(N, 16 * RT)), dim3(64 * KS), \
                               0, st, E, COUNT, LIST, XIN, w.cell2, SH, G.W2, WL, HL, w.HR,         \
                               pk.po[LI], L[LI].ln_gamma, L[LI].ln_beta, XOUT);                     \
    } while (0)
    const int *const n2_dev = w.counts + 0, *const n3_dev = w.counts + 1;
    OUTT(0, SSLA_C1, SSLA_C2, 2, 1, 3, kOutKSFew, E, no_count, no_list, w.X0, 0, G.W2, G.H2, w.X1);
    MARK();
    // ---- [side] the s3 record order, tdrop_s3, s3 pair and group tables ---
    // (enqueued after L4's launches: the host needs a few microseconds per
    // launch, and L4 keeps the device busy meanwhile)
    if (!small_all) {
        hipLaunchKernelGGL(k_keys3a, dim3(grid1(nk3, 256)), dim3(256), 0, s3, nk3, G, w.n2, w.bd,
                           w.t3, w.n3);
        hipLaunchKernelGGL((k_keyscan<false, false>), dim3(1), dim3(kScanThreads), 0, s3, (int)nk3, w.t3,
                           w.st3, w.en3, (int*)nullptr, w.n3, w.off3, w.counts + 1, KeyHist{},
                           GroupTab{});
        hipLaunchKernelGGL(k_place3, dim3(grid1(nmax2, 256)), dim3(256), 0, s3, (const int*)(w.counts + 0),
                           w.list2, w.bd, G, w.cell2, w.sidx, V2, w.st2, w.en2, w.old2, w.st3, K3, V3,
                           w.key3g);
        hipLaunchKernelGGL(k_tdrop3, dim3(grid1(nmax2, 256)), dim3(256), 0, s3, (const int*)(w.counts + 0),
                           K3, V3, nk3, G.C3, w.st3, w.off3, w.bd, G.window, w.owner,
                           have_head ? 1 : 0, w.pass3, w.list3, w.last3, w.cnt3);
        hipLaunchKernelGGL(k_keys3b, dim3(grid1(nk3, 256)), dim3(256), 0, s3, nk3, G, w.t3, w.bd,
                           w.pcnt);
        if (gt3) {
            hipLaunchKernelGGL((k_keyscan<false, true>), dim3(1), dim3(kScanThreads), 0, s3, (int)nk3,
                               w.pcnt, w.pst3, (int*)nullptr, w.goff3, (const int*)nullptr, (int*)nullptr,
                               (int*)nullptr, KeyHist{}, GroupTab{nv, w.glist3, w.counts + 7});
        } else {
            hipLaunchKernelGGL((k_keyscan<false, false>), dim3(1), dim3(kScanThreads), 0, s3, (int)nk3,
                               w.pcnt, w.pst3, (int*)nullptr, w.goff3, (const int*)nullptr, (int*)nullptr,
                               (int*)nullptr, KeyHist{}, GroupTab{});
            hipLaunchKernelGGL(k_key_groups, dim3(grid1(nk3, 256)), dim3(256), 0, s3, nk3, w.pst3, w.gcnt3,
                               w.gend3, w.ghist3, w.gw3);
            hipLaunchKernelGGL(k_group_order, dim3(1), dim3(kScanThreads), 0, s3, (int)nk3, nv, w.pst3,
                               w.goff3, w.gcnt3, w.gend3, w.ghist3, w.gw3, w.gstart3, w.gbase3, w.glist3,
                               w.counts + 7);
        }
#define PAIR_RANK3(SMALL)                                                                             \
    hipLaunchKernelGGL(k_pair_rank<SMALL>, dim3(grid1(nmax2, 256)), dim3(256), 0, s3, E, n2_dev, K3, V3, nk3, \
                       G.C3, G.W3, G.H3, w.st3, w.en3, w.pst3, w.pent3, w.pass3)
        if (nmax2 <= kSmallRec) PAIR_RANK3(true);
        else PAIR_RANK3(false);
#undef PAIR_RANK3
        HIPCHK(hipEventRecord(w.s3_ordered, s3));
    }
    HIPCHK(hipGetLastError());
    // ---- L5: 48 -> 48, state for all records, output for pass2 ---------------
    PSCAN(SSLA_C2, SSLA_C2, true, 1, 2, 6, w.glist, false, w.X1, G.C2, gridS4);
    OUTT(1, SSLA_C2, SSLA_C2, kOutRT5, kOutKS5, 1, kOutKSFew, nmax2, n2_dev, w.list2, w.X1, 0, G.W2, G.H2, w.X2);
    MARK();
    // ---- L6: 48 -> 96, pass2 records ------------------------------------------
    if (!small_all) HIPCHK(hipStreamWaitEvent(st, w.s3_ordered, 0));
    PSCAN(SSLA_C2, SSLA_C3, false, 2, 3, 7, w.glist3, true, w.X2, G.C3, gridS6);
    OUTT(2, SSLA_C2, SSLA_C3, kOutRT6, kOutKS6, 1, kOutKSFew, nmax2, n2_dev, w.list2, w.X2, 1, G.W3, G.H3, w.X3);
    MARK();
    // ---- L7: 96 -> 96, state for pass2, output for pass3 ----------------------
    PSCAN(SSLA_C3, SSLA_C3, false, 3, 3, 7, w.glist3, false, w.X3, G.C3, gridS6);
    OUTT(3, SSLA_C3, SSLA_C3, kOutRT7, kOutKS7, 1, kOutKSFew7, nmax3, n3_dev, w.list3, w.X3, 1, G.W3, G.H3, w.X4);
    MARK();
    HIPCHK(hipGetLastError());
    // ---- head ------------------------------------------------------------------
    if (have_head) {
        const HeadPtrs hp = head_ptrs(cfg);
        const PredGrid pg{w.owner, w.key3g, w.last3, w.cnt3, w.bd, G};
        if (head == kHeadYolox)
            hipLaunchKernelGGL(k_head, dim3(tiles3), dim3(kHeadThreads), 0, st, (const int*)(w.counts + 1),
                               w.list3, w.X4, hp, pg, w.H7);
        else
            hipLaunchKernelGGL(k_head_linear, dim3(tiles3), dim3(256), 0, st,
                               (const int*)(w.counts + 1), w.list3, w.X4, hp, pg, w.H7);
    }
    MARK();
    if (grid1(E, kEmitRec) < cus)
        hipLaunchKernelGGL(k_emit<kEmitRecFew>, dim3(grid1(E, kEmitRecFew)), dim3(256), 0, st, E, w.bd, nb,
                           w.cell2, w.owner, w.pass2, w.pass3, w.X4, w.H7, have_head ? 1 : 0);
    else
        hipLaunchKernelGGL(k_emit<kEmitRec>, dim3(grid1(E, kEmitRec)), dim3(256), 0, st, E, w.bd, nb, w.cell2,
                           w.owner, w.pass2, w.pass3, w.X4, w.H7, have_head ? 1 : 0);
    HIPCHK(hipGetLastError());
    MARK();
#undef MARK
#undef PSCAN
#undef OUTT
    end.finish();
    if (phase_ms) {
        // this call's events join the pending ones (read below when sync is
        // set, else by a later call with sync)
        if (w.pending.size() >= kMaxPending) {
            const int rc = flush_pending(w, 1);
            if (rc) return rc;
        }
        Workspace::Pending p;
        for (int k = 0; k <= SSLA_DRAIN_PHASES; ++k) {
            p.ev[k] = ev[k];
            ev[k] = nullptr;
        }
        p.phase_ms = phase_ms;
        p.pmask = pmask;
        w.pending.push_back(p);
    }
    if (sync) {
        HIPCHK(hipStreamSynchronize(st));
        if (__atomic_exchange_n(w.scan_err, 0, __ATOMIC_RELAXED)) {
            set_error("drain: a wait of the recurrence's look-back ran out (results are invalid)");
            return SSLA_ERR_HIP;
        }
        // every earlier call finished before this one's kernels started
        const int rc = flush_pending(w, w.pending.size());
        if (rc) return rc;
    }
    return SSLA_OK;
}

}  // namespace ssla
