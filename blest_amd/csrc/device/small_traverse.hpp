// One workgroup traverses one small symmetric graph (n <= 131072) over its CSR, with the
// visited / frontier / next bitmaps in LDS: the graph batch (a workgroup per graph) and the
// single-source BFS of a graph small enough that level kernels cost more than the work.
#pragma once

#include "dev_common.hpp"

namespace blest {
namespace dev {

// What bounds such a traversal is not bandwidth (a graph's 2 MB of lists are read about once) but
// the round trips of dependent loads: list bounds, list entries, one after another, in one
// workgroup.  Hence 32 waves per CU (two graphs), and in every step as many independent
// loads as the registers of 8 waves per SIMD hold:
//   top-down   the frontier vertices of 64 bitmap words are dealt out to the lanes one each
//              (a sparse frontier fills whole waves), kBatchTd list entries per step;
//   bottom-up  a lane takes its vertex of kBatchWords words at once, kBatchBu entries of
//              each per step; found vertices go straight into visited and next;
//   a list still open after kBatchOwn entries is finished by its whole wave;
//   graphs of at most 65536 vertices keep 16-bit list entries (635 -> 560 us below), and
//   the switch to bottom-up waits until the frontier's edges are a quarter of the open
//   ones (alpha 4): a top-down discovery is an LDS atomic, while a bottom-up sweep reads
//   every line of the lists (alpha 15: 560 us, 8: 490, 4: 440, 2: 440).
// Measured (MI355X), 512 Erdos-Renyi graphs, n ~ U[1024, 65536], degree 8: 2.06 ms with a
// wave per rset (16 lanes busy at degree 8) and a lane walking one vertex's list entry by
// entry, 0.37 ms in this form (4 words 0.40, 8 entries of 4 words spill: 0.55).
constexpr int kBatchBlock = 1024;
constexpr int kBatchTd = 8, kBatchWords = 3, kBatchBu = 4;
constexpr uint32_t kBatchOwn = 32;

// N list entries as one load per 16 bytes.  A CU's vector cache takes about one line per
// clock, so entry-wise loads of 64 lists cost a line access per entry (628 us for 512 graphs
// of 65536 vertices, 575 us with these); lists start at any entry, which unaligned vector
// loads take, and the list array is padded by a step's length past its last entry.
template <class Idx, int N>
struct __attribute__((packed, aligned(sizeof(Idx)))) ListStep {
    Idx v[N];
};
template <int N, class Idx>
__device__ __forceinline__ ListStep<Idx, N> load_step(const Idx* ci, uint32_t p) {
    return *reinterpret_cast<const ListStep<Idx, N>*>(ci + p);
}

// Position of the k-th (from 0) set bit of x; x has more than k bits.
__device__ __forceinline__ unsigned nth_bit(unsigned long long x, unsigned k) {
    unsigned pos = 0;
#pragma unroll
    for (int width = 32; width > 0; width >>= 1) {
        const unsigned c = __popcll((x >> pos) & ((1ull << width) - 1));
        if (k >= c) {
            k -= c;
            pos += width;
        }
    }
    return pos;
}

struct SmallGraph {
    uint32_t n;
    const uint32_t* cp;  // n + 1 list offsets
};

// Totals of a traversal (every thread gets them).
struct SmallTotals {
    unsigned levels, visited, td, bu;
    unsigned long long edges, buMask;
};

// The whole workgroup (kBatchBlock threads) traverses G from src; ci: its lists, readable
// one step past the last entry.  bitmaps: 3 x words of LDS; sNew / sEdges: vertices
// discovered by level (slot L % 3) and their degree sum.  Levels go to `levels` (-1 where
// unreached), complete for the workgroup after the next barrier.
template <class Idx>
__device__ __forceinline__ SmallTotals small_traverse(const SmallGraph& G, uint32_t src, const Idx* ci,
                                                      int32_t* levels, double alpha, double beta,
                                                      unsigned long long* bitmaps, uint32_t words, unsigned* sNew,
                                                      unsigned long long* sEdges) {
    const uint32_t n = G.n, W = (n + 63) / 64;
    unsigned long long* vis = bitmaps;
    unsigned long long* front = bitmaps + words;
    unsigned long long* next = bitmaps + 2 * words;
    const uint32_t* cp = G.cp;
    SmallTotals tot{0, 0, 0, 0, 0, 0};
    const unsigned lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    constexpr unsigned nwaves = kBatchBlock / kWave;
    for (uint32_t w = threadIdx.x; w < W; w += kBatchBlock) {
        const unsigned long long x = (w == src / 64) ? (1ull << (src & 63)) : 0ull;
        vis[w] = x;
        front[w] = x;
        next[w] = 0ull;
    }
    if (threadIdx.x == 0) {
        levels[src] = 0;
        sNew[0] = 1;
        sEdges[0] = cp[src + 1] - cp[src];
        sNew[1] = 0;
        sEdges[1] = 0;
    }
    __syncthreads();
    const unsigned long long m = cp[n];
    bool bottomUp = false, clean = true;  // clean: next is all zero
    for (unsigned L = 1;; ++L) {
        const unsigned nf = sNew[(L - 1) % 3];
        const unsigned long long mf = sEdges[(L - 1) % 3];
        if (nf == 0) break;
        tot.levels = L;
        tot.visited += nf;
        tot.edges += mf;
        if (!bottomUp && double(mf) * alpha > double(m - min(tot.edges, m))) bottomUp = true;
        else if (bottomUp && double(nf) * beta < double(n)) bottomUp = false;
        tot.td += bottomUp ? 0u : 1u;
        tot.bu += bottomUp ? 1u : 0u;
        if (bottomUp && L <= 64) tot.buMask |= 1ull << (L - 1);
        if (threadIdx.x == 0) {  // last read at the top of the level before, a barrier ago
            sNew[(L + 1) % 3] = 0;
            sEdges[(L + 1) % 3] = 0;
        }
        unsigned cnt = 0;
        unsigned long long edges = 0;
        if (!bottomUp) {
            if (!clean) {
                for (uint32_t w = threadIdx.x; w < W; w += kBatchBlock) next[w] = 0ull;
                __syncthreads();
            }
            const uint32_t* vis32 = reinterpret_cast<const uint32_t*>(vis);
            uint32_t* next32 = reinterpret_cast<uint32_t*>(next);
            auto reach = [&](uint32_t u) {
                const uint32_t bit = 1u << (u & 31);
                if (!(vis32[u >> 5] & bit)) atomicOr(&next32[u >> 5], bit);
            };
            // words wave, wave + nwaves, ...: 64 of them at a time, word i0 + lane per lane
            for (uint32_t i0 = 0; i0 * nwaves + wave < W; i0 += kWave) {
                const uint32_t w = (i0 + lane) * nwaves + wave;
                const unsigned long long f = w < W ? front[w] : 0ull;
                const unsigned c = __popcll(f);
                const unsigned incl = wave_inclusive_scan(c), excl = incl - c;
                const unsigned total = __shfl(incl, kWave - 1, kWave);
                for (unsigned t0 = 0; t0 < total; t0 += kWave) {
                    const unsigned t = t0 + lane;
                    const unsigned owner = wave_owner(excl, min(t, total - 1));
                    const unsigned long long of = __shfl(f, owner, kWave);
                    const unsigned oex = __shfl(excl, owner, kWave);
                    uint32_t p = 0, e = 0;
                    if (t < total) {
                        const uint32_t v = ((i0 + owner) * nwaves + wave) * 64 + nth_bit(of, t - oex);
                        p = cp[v];
                        e = cp[v + 1];
                    }
                    const uint32_t own = min(e, p + kBatchOwn);
                    while (p < own) {
                        const auto step = load_step<kBatchTd>(ci, p);
#pragma unroll
                        for (int j = 0; j < kBatchTd; ++j) reach(p + j < own ? uint32_t(step.v[j]) : src);  // src: visited
                        p += kBatchTd;
                    }
                    p = own;
                    for (unsigned long long h = __ballot(p < e); h; h &= h - 1) {
                        const int l = __builtin_ctzll(h);
                        const uint32_t hp = __shfl(p, l, kWave), he = __shfl(e, l, kWave);
                        for (uint32_t q0 = hp; q0 < he; q0 += 4 * kWave) {
                            uint32_t u[4];
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                const uint32_t q = q0 + j * kWave + lane;
                                u[j] = q < he ? uint32_t(ci[q]) : src;
                            }
#pragma unroll
                            for (int j = 0; j < 4; ++j) reach(u[j]);
                        }
                    }
                }
            }
            __syncthreads();
            // fold: lane per vertex; the spent frontier becomes the next level's empty `next`
            for (uint32_t w0 = wave; w0 < W; w0 += nwaves * kBatchWords) {
                unsigned long long nw[kBatchWords];
                uint32_t lo[kBatchWords], hi[kBatchWords];
#pragma unroll
                for (int k = 0; k < kBatchWords; ++k) {
                    const uint32_t w = w0 + k * nwaves, v = w * 64 + lane;
                    nw[k] = w < W ? next[w] : 0ull;
                    lo[k] = hi[k] = 0;
                    if ((nw[k] >> lane) & 1ull) {
                        lo[k] = cp[v];
                        hi[k] = cp[v + 1];
                        levels[v] = int32_t(L);
                        ++cnt;
                    }
                    if (lane == 0 && w < W) {
                        vis[w] |= nw[k];
                        front[w] = 0ull;
                    }
                }
#pragma unroll
                for (int k = 0; k < kBatchWords; ++k) edges += hi[k] - lo[k];
            }
            clean = true;
        } else {
            const uint32_t* front32 = reinterpret_cast<const uint32_t*>(front);
            for (uint32_t w0 = wave; w0 < W; w0 += nwaves * kBatchWords) {
                uint32_t b[kBatchWords], e[kBatchWords];
                unsigned open = 0, found = 0;  // bit k: the vertex of word k
#pragma unroll
                for (int k = 0; k < kBatchWords; ++k) {
                    const uint32_t w = w0 + k * nwaves, v = w * 64 + lane;
                    const bool o = w < W && v < n && !((vis[min(w, W - 1)] >> lane) & 1ull);
                    b[k] = o ? cp[v] : 0u;
                    e[k] = o ? cp[v + 1] : 0u;
                }
#pragma unroll
                for (int k = 0; k < kBatchWords; ++k)
                    if (b[k] < e[k]) open |= 1u << k;
                for (uint32_t off = 0; off < kBatchOwn && __ballot(open != 0); off += kBatchBu) {
                    ListStep<Idx, kBatchBu> u[kBatchWords];
#pragma unroll
                    for (int k = 0; k < kBatchWords; ++k)
                        if ((open >> k) & 1u) u[k] = load_step<kBatchBu>(ci, b[k] + off);
#pragma unroll
                    for (int k = 0; k < kBatchWords; ++k) {
                        if ((open >> k) & 1u) {
                            bool hit = false;
#pragma unroll
                            for (int j = 0; j < kBatchBu; ++j)
                                if (b[k] + off + j < e[k]) hit |= (front32[u[k].v[j] >> 5] >> (u[k].v[j] & 31)) & 1u;
                            if (hit) found |= 1u << k;
                            if (hit || b[k] + off + kBatchBu >= e[k]) open &= ~(1u << k);
                        }
                    }
                }
#pragma unroll
                for (int k = 0; k < kBatchWords; ++k) {
                    for (unsigned long long h = __ballot((open >> k) & 1u); h; h &= h - 1) {
                        const int l = __builtin_ctzll(h);
                        const uint32_t hp = __shfl(b[k], l, kWave) + kBatchOwn, he = __shfl(e[k], l, kWave);
                        bool hit = false;
                        for (uint32_t q0 = hp; q0 < he && !hit; q0 += kWave) {  // wave-uniform
                            const uint32_t q = q0 + lane;
                            const uint32_t u = ci[min(q, he - 1)];
                            hit = __ballot(q < he && ((front32[u >> 5] >> (u & 31)) & 1u)) != 0ull;
                        }
                        if (hit && lane == unsigned(l)) found |= 1u << k;
                    }
                    const uint32_t w = w0 + k * nwaves;
                    const bool f = (found >> k) & 1u;
                    const unsigned long long fw = __ballot(f);
                    if (f) {
                        levels[w * 64 + lane] = int32_t(L);
                        ++cnt;
                        edges += e[k] - b[k];
                    }
                    if (lane == 0 && w < W) {
                        next[w] = fw;
                        if (fw) vis[w] |= fw;  // this wave's word alone
                    }
                }
            }
            clean = false;  // the spent frontier becomes `next`
        }
        cnt = wave_sum_u32(cnt);
        edges = wave_sum_u64(edges);
        if (lane == 0 && cnt) {
            atomicAdd(&sNew[L % 3], cnt);
            atomicAdd(&sEdges[L % 3], edges);
        }
        __syncthreads();
        unsigned long long* spent = front;
        front = next;
        next = spent;
    }
    for (uint32_t w = wave; w < W; w += nwaves) {
        const uint32_t v = w * 64 + lane;
        if (v < n && !((vis[w] >> lane) & 1ull)) levels[v] = -1;
    }
    return tot;
}

}  // namespace dev
}  // namespace blest
