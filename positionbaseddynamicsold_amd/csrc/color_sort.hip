// Constraint-graph colouring and a stable LDS radix-sort pass (gfx950).
//
// Colouring follows the reference's bulk-synchronous speculative scheme:
// AssignColorsGPU (PBD_cuda.cu:313-372) then ResolveConflictsGPU (:374-431),
// repeated until every prim is coloured.  Assign reads `color` and writes
// `prd` only for uncoloured prims; resolve reads `prd` and writes `color` of
// its own prim only, so each pass sees the previous pass's arrays and the
// result does not depend on scheduling.  Unlike the reference (a fixed 20000
// rounds, PBD_cuda.cu:508,826) the host stops as soon as no prim is left
// uncoloured.
#include "pbd_internal.hpp"

namespace pbd {

__global__ __launch_bounds__(256) void k_color_assign(const int2* __restrict__ adj_sn,
                                                      const int* __restrict__ adj,
                                                      const int* __restrict__ color,
                                                      int* __restrict__ prd, int np) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    if (color[p] >= 0) return;
    int2 sn = adj_sn[p];
    int c = -1, offset = 0;
    while (c < 0) {
        unsigned long long forbidden = 0ull;
        for (int i = sn.x; i < sn.x + sn.y; ++i) {
            int nc = color[adj[i]] - offset;
            if (nc >= 0 && nc < 64) forbidden |= (1ull << nc);
        }
        if (forbidden != ~0ull) {
            // first zero bit == log2((~x) & (x+1)) of the reference
            c = offset + __builtin_ctzll(~forbidden);
        } else {
            offset += 64;
        }
    }
    prd[p] = c;
}

// Keeps the proposal of every prim that has no conflicting neighbour of
// higher priority (more points, then lower id); the prims left uncoloured
// are counted into *uncolored with one atomic per workgroup (one per wave
// had the atomics on that one address take most of the round).
__global__ __launch_bounds__(256) void k_color_resolve(const int* __restrict__ npts,
                                                       const int2* __restrict__ adj_sn,
                                                       const int* __restrict__ adj,
                                                       int* __restrict__ color,
                                                       const int* __restrict__ prd, int np,
                                                       int* __restrict__ uncolored) {
    __shared__ int wave_left[4];
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    int left = 0;
    if (p < np && color[p] < 0) {
        int2 sn = adj_sn[p];
        int c = prd[p], conflict = 0, npt = npts[p];
        for (int i = sn.x; i < sn.x + sn.y; ++i) {
            int n = adj[i];
            if (prd[n] == c) {
                int nnpt = npts[n];
                if (nnpt > npt || (nnpt == npt && n < p)) {
                    conflict = 1;
                    break;
                }
            }
        }
        if (conflict) left = 1;
        else color[p] = c;
    }
    const unsigned long long m = __ballot(left);
    if ((threadIdx.x & 63) == 0) wave_left[threadIdx.x >> 6] = (int)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        const int tot = wave_left[0] + wave_left[1] + wave_left[2] + wave_left[3];
        if (tot) atomicAdd(uncolored, tot);
    }
}

int launch_color_round(hipStream_t s, const int* npts, const int* adj_sn, const int* adj, int* color, int* prd,
                       int* uncolored, int np) {
    int nb = (np + 255) / 256;
    if (nb == 0) return 0;
    hipLaunchKernelGGL(k_color_assign, dim3(nb), dim3(256), 0, s, (const int2*)adj_sn, adj, color, prd, np);
    hipLaunchKernelGGL(k_color_resolve, dim3(nb), dim3(256), 0, s, npts, (const int2*)adj_sn, adj, color, prd,
                       np, uncolored);
    PBD_HIP(hipGetLastError());
    return 0;
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort of (key, value) uint32 pairs, 8-bit digits.  A pass is
// two launches over tiles of 4096 consecutive elements: k_radix_hist counts
// digit d of tile b into counts[b * 256 + d]; k_radix_scatter sums the rows of
// the tiles before its own (and of all tiles, for the digits before) itself,
// ranks equal digits of its tile in input order (wave match, per-wave counts)
// and writes.  With more than RADIX_ROWS tiles the sums come from a launch of
// their own (k_radix_rows).  Launches and their latencies bound the sort: half
// a million pairs are 4 MB, a microsecond of bandwidth, per pass, which took
// 37 us with a scan of three launches and a workgroup barrier per 256
// elements, 16 us so.
// ---------------------------------------------------------------------------
constexpr int RB = RADIX_TILE, RT = 1024, RW = RT / 64, RR = RB / RT;
constexpr int RADIX_ROWS = 256;

__global__ __launch_bounds__(RT) void k_radix_hist(const uint32_t* __restrict__ keys, int n, int shift,
                                                   int* __restrict__ counts) {
    __shared__ int h[256];
    const int t = threadIdx.x;
    if (t < 256) h[t] = 0;
    uint32_t k[RR];
    for (int r = 0; r < RR; r++) {
        const int i = blockIdx.x * RB + r * RT + t;
        k[r] = i < n ? keys[i] : 0u;
    }
    __syncthreads();
    for (int r = 0; r < RR; r++)
        if (blockIdx.x * RB + r * RT + t < n) atomicAdd(&h[(k[r] >> shift) & 255u], 1);
    __syncthreads();
    if (t < 256) counts[blockIdx.x * 256 + t] = h[t];
}

// rows[b][d] = digit d's count in the tiles before b, rows[nb][d] in all; one
// workgroup per digit.
__global__ __launch_bounds__(256) void k_radix_rows(const int* __restrict__ counts, int nb, int* __restrict__ rows) {
    __shared__ int wave[4];
    const int d = blockIdx.x, t = threadIdx.x, lane = t & 63, wv = t >> 6;
    int carry = 0;
    for (int b0 = 0; b0 < nb; b0 += 256) {
        const int b = b0 + t, c = b < nb ? counts[(size_t)b * 256 + d] : 0;
        int run = c;
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(run, off);
            if (lane >= off) run += o;
        }
        if (lane == 63) wave[wv] = run;
        __syncthreads();
        for (int w = 0; w < wv; w++) run += wave[w];
        if (b < nb) rows[(size_t)b * 256 + d] = carry + run - c;
        carry += wave[0] + wave[1] + wave[2] + wave[3];
        __syncthreads();
    }
    if (t == 0) rows[(size_t)nb * 256 + d] = carry;
}

// rows: from k_radix_rows, or nullptr: summed from counts here.  vin nullptr:
// the values are the positions.  Keys are written less `less`.
__global__ __launch_bounds__(RT) void k_radix_scatter(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                      uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, int n,
                                                      int shift, const int* __restrict__ counts,
                                                      const int* __restrict__ rows, int nb, uint32_t less) {
    __shared__ int wcnt[RW][256];
    __shared__ int before[RT / 256][256], all[RT / 256][256], start[256], base[256], wave[4], here[4];
    __shared__ uint2 tile[RB];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, b = blockIdx.x;
    // this wave's elements, in order
    const int i0 = b * RB + wv * (RB / RW) + lane;
    uint32_t k[RR], v[RR];
    for (int r = 0; r < RR; r++) {
        const int i = i0 + 64 * r;
        k[r] = i < n ? kin[i] : 0u;
        v[r] = i < n ? (vin ? vin[i] : (uint32_t)i) : 0u;
    }
    {
        const int d = t & 255, part = t >> 8;
        int pre = 0, sum = 0;
        if (rows) {
            if (part == 0) {
                pre = rows[(size_t)b * 256 + d];
                sum = rows[(size_t)nb * 256 + d];
            }
        } else {
            for (int q0 = part; q0 < nb; q0 += 16 * (RT / 256)) {
                int c[16];  // in flight together
#pragma unroll
                for (int u = 0; u < 16; u++) c[u] = counts[min(q0 + u * (RT / 256), nb - 1) * 256 + d];
#pragma unroll
                for (int u = 0; u < 16; u++) {
                    const int q = q0 + u * (RT / 256);
                    sum += q < nb ? c[u] : 0;
                    pre += q < b ? c[u] : 0;
                }
            }
        }
        before[part][d] = pre;
        all[part][d] = sum;
        for (int j = t; j < RW * 256; j += RT) (&wcnt[0][0])[j] = 0;
    }
    __syncthreads();
    int rank[RR];
    for (int r = 0; r < RR; r++) {
        const bool valid = i0 + 64 * r < n;
        const int d = (k[r] >> shift) & 255u;
        // lanes with this lane's digit: one ballot per digit bit, so the cost
        // does not depend on how many distinct digits the wave holds
        unsigned long long m = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; bit++) {
            const bool set = (d >> bit) & 1;
            const unsigned long long bb = __ballot(valid && set);
            m &= set ? bb : ~bb;
        }
        const int below = __popcll(m & __lanemask_lt());
        if (valid) {
            rank[r] = wcnt[wv][d] + below;
            __builtin_amdgcn_wave_barrier();  // read before the digit's first lane adds
            if (below == 0) wcnt[wv][d] = rank[r] + __popcll(m);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // digit starts, and each wave's place within its digit
    int pre = 0, sum = 0, incl = 0, mine = 0, upto = 0;  // digit t in all tiles and in this one
    if (t < 256) {
        for (int q = 0; q < RT / 256; q++) {
            pre += before[q][t];
            sum += all[q][t];
        }
        incl = sum;
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(incl, off);
            if (lane >= off) incl += o;
        }
        if (lane == 63) wave[wv] = incl;
        for (int w = 0; w < RW; w++) {
            const int c = wcnt[w][t];
            wcnt[w][t] = mine;
            mine += c;
        }
        upto = mine;
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(upto, off);
            if (lane >= off) upto += o;
        }
        if (lane == 63) here[wv] = upto;
    }
    __syncthreads();
    if (t < 256) {
        for (int w = 0; w < wv; w++) {
            incl += wave[w];
            upto += here[w];
        }
        start[t] = upto - mine;
        base[t] = incl - sum + pre - start[t];
    }
    __syncthreads();
    // in order in LDS first, so that the stores of a wave run over a few digits' places
    for (int r = 0; r < RR; r++)
        if (i0 + 64 * r < n) {
            const int d = (k[r] >> shift) & 255u;
            tile[start[d] + wcnt[wv][d] + rank[r]] = make_uint2(k[r], v[r]);
        }
    __syncthreads();
    const int m = min(RB, n - b * RB);
    for (int i = t; i < m; i += RT) {
        const uint2 e = tile[i];
        const int pos = base[(e.x >> shift) & 255u] + i;
        kout[pos] = e.x - less;
        vout[pos] = e.y;
    }
}

// Stable sort of n (key, value) pairs on bits [0, bits) of the key from src
// into out by way of tmp; src may be tmp when radix_passes(bits) is odd, out
// when it is even.  sv == nullptr: the values are 0 .. n - 1.  counted: the
// first digit's counts are in hist.  Keys come out less `less`.
void radix_sort(hipStream_t s, const uint32_t* sk, const uint32_t* sv, uint32_t* tk, uint32_t* tv, uint32_t* ok,
                uint32_t* ov, int n, int bits, int* hist, bool counted, uint32_t less) {
    if (n <= 0) return;
    const int nb = radix_tiles(n), passes = radix_passes(bits);
    int* rows = nb > RADIX_ROWS ? hist + (size_t)256 * nb : nullptr;
    for (int ps = 0; ps < passes; ps++) {
        const bool last = ps + 1 == passes, to_out = (passes - 1 - ps) % 2 == 0;
        if (ps > 0 || !counted) hipLaunchKernelGGL(k_radix_hist, dim3(nb), dim3(RT), 0, s, sk, n, ps * 8, hist);
        if (rows) hipLaunchKernelGGL(k_radix_rows, dim3(256), dim3(256), 0, s, hist, nb, rows);
        uint32_t *k = to_out ? ok : tk, *v = to_out ? ov : tv;
        hipLaunchKernelGGL(k_radix_scatter, dim3(nb), dim3(RT), 0, s, sk, sv, k, v, n, ps * 8, hist, rows, nb,
                           last ? less : 0u);
        sk = k;
        sv = v;
    }
    PBD_HIP(hipGetLastError());
}

// In place, with (k2, v2) as the other buffer.
void radix_sort_pairs(hipStream_t s, uint32_t* k, uint32_t* v, uint32_t* k2, uint32_t* v2, int n, int bits, int* hist) {
    if (n <= 0) return;
    if (radix_passes(bits) % 2 == 0) return radix_sort(s, k, v, k2, v2, k, v, n, bits, hist, false, 0u);
    radix_sort(s, k, v, k, v, k2, v2, n, bits, hist, false, 0u);
    PBD_HIP(hipMemcpyAsync(k, k2, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, s));
    PBD_HIP(hipMemcpyAsync(v, v2, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, s));
}

}  // namespace pbd
