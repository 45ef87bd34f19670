// Backward of the fused d/D outputs: the gradients of positions and cell
// from the gradients of D (pairs x 3) and d (pairs), for the pairs written by
// the emitting kernels.  It replaces the autograd of the reference's Torch
// expression (src/tonari/_torch_frontend.py:92-104)
//   D_e = pos[j_e] - pos[i_e] + S_e @ cell[b_e],   d_e = |D_e|,
// whose gradient is, with g_e = dL/dD_e + dL/dd_e * D_e / d_e (0 when
// d_e = 0, as torch's vector_norm backward):
//   dL/dpos[j_e] += g_e,  dL/dpos[i_e] -= g_e,  dL/dcell[b_e][a][c] += S_e[a] g_e[c].
//
// Each wave takes a contiguous range of pairs, two per lane and round; the
// next round's rows load while the current ones are summed.
// Position gradients are summed in an LDS table of the workgroup and added
// to grad_pos once per atom at the end.  What bounds the kernel otherwise is
// the rate of global float atomics: about 21 G cache-line requests per
// second, whatever the type, where lanes that touch one line in one
// instruction cost one request (4 M random 12-byte triples: 586 us with
// three instructions per lane, 220 us with three lanes per triple).
// Therefore every global add is made by three neighbouring lanes.
//   Direct table: when the atoms of the structures of the workgroup's pairs
//   fit the table, an atom's slot is its distance from the first of them.
//   Hashed table (larger structures): open addressing, keyed by atom; the
//   atoms of consecutive pairs are few when the list comes in bin order (a
//   few hundred stencil atoms for some thousand pairs).  Atoms that find no
//   slot within kBwdProbes probes are added to grad_pos directly.
// The pairs of a source are contiguous: its side is a segmented sum over
// the round's lanes (DPP, no LDS), one table add per run.  The pairs of a
// structure are contiguous too (sources come in index or bin order, both
// grouped by structure), so each wave keeps the atom range of its current
// structure and per-lane partial cell sums, reduces them when a source
// leaves that range, and the waves of a block merge their last sums: a
// structure's 9 entries take a few atomics per block, not per pair.  Float
// atomics make the summation order vary between runs (the same holds for
// torch's index_add on the device).
//
// Measured on the MI355X, before (one round in flight, a table of the input
// type, 8,192 pairs per workgroup whatever the list, a binary search of
// batch_ptr per pair) and now: 9.05 M float32 pairs in bin order, gradient of
// D, 329 -> 117 us alone, back to back (3.1 TB/s; streaming the rows alone
// takes 62; 137 in a step, behind an emit's write-backs); 1.6 M pairs
// of 256 small crystals 110 -> 22 us; 17 k float64 pairs of 512 atoms 37 ->
// 8 us; 37 M float64 pairs of slabs in index order, gradient of d, 4.38 ->
// 1.9 ms, and 0.52 ms with their sources' runs (k_geometry_backward_runs).
#pragma once

#include "nl_query.h"

namespace tnr {

constexpr int kBwdBlock = 512;
constexpr int kBwdWaves = kBwdBlock / kWave;
constexpr int kBwdSlots = 2048;  // LDS slots per workgroup (power of two)
constexpr int kBwdProbes = 8;
constexpr int kBwdRows = 2;      // pairs per lane and round

// Pairs of each wave's range: whole rounds of 64 kBwdRows, so many that a
// list of up to 2 M pairs makes about 2,048 waves (the device holds 4,096;
// fewer pairs per wave mean more atoms flushed per pair), and at most 8
// rounds: 8,192 pairs per workgroup, whose atoms fill about half the hashed
// table when 90 neighbours of each source lie in its bin's stencil.  The
// 100,000-atom float32 list, gradient of D, alone: 110 us at 8 rounds, 114 at 4,
// 146 at 16 (too few workgroups), 131 with one pair per lane.
// The grid and the kernel both take the range from here.
inline int64_t backward_pairs_per_wave(int64_t n_pairs) {
    constexpr int64_t round = kWave * kBwdRows, most = 8, waves = 2048;
    const int64_t rounds = (n_pairs + round - 1) / round;
    const int64_t r = (rounds + waves - 1) / waves;
    return round * (r < 1 ? 1 : r > most ? most : r);
}

// x of the lane that CTRL names in the rows of ROWS, 0 where there is none.
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_value(float x) {
    return __int_as_float(dpp_move<CTRL, ROWS>(__float_as_int(x)));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_value(double x) {
    return __hiloint2double(dpp_move<CTRL, ROWS>(__double2hiint(x)),
                            dpp_move<CTRL, ROWS>(__double2loint(x)));
}

// Sum over the wave, valid in lane 63.
template <typename T>
__device__ __forceinline__ T wave_sum(T x) {
    x += dpp_value<0x111, 0xf>(x);
    x += dpp_value<0x112, 0xf>(x);
    x += dpp_value<0x114, 0xf>(x);
    x += dpp_value<0x118, 0xf>(x);
    x += dpp_value<0x142, 0xa>(x);
    x += dpp_value<0x143, 0xc>(x);
    return x;
}

// Inclusive sums within segments of consecutive lanes: x gains the sums of
// the lanes from the segment's first lane seg0 on.  `near` = lane - seg0.
template <typename T>
__device__ __forceinline__ void segment_sums(T (&x)[3], int seg0, int lane) {
    const int near = lane - seg0;
    const int row = lane & 15;
    const bool c1 = near >= 1, c2 = near >= 2, c4 = near >= 4, c8 = near >= 8;
    // the segment reaches into the row (the half wave) before the lane's
    const bool c15 = near > row, c31 = near > (lane & 31);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        T y = dpp_value<0x111, 0xf>(x[c]);
        x[c] += c1 ? y : T(0);
        y = dpp_value<0x112, 0xf>(x[c]);
        x[c] += c2 ? y : T(0);
        y = dpp_value<0x114, 0xf>(x[c]);
        x[c] += c4 ? y : T(0);
        y = dpp_value<0x118, 0xf>(x[c]);
        x[c] += c8 ? y : T(0);
        y = dpp_value<0x142, 0xa>(x[c]);
        x[c] += c15 ? y : T(0);
        y = dpp_value<0x143, 0xc>(x[c]);
        x[c] += c31 ? y : T(0);
    }
}

// One pair's row as loaded.
// (source and target by two 4-byte loads: of a 16-byte load the unused
// halves' registers are taken for other values at once, which waits for it)
template <typename T>
struct BwdRow {
    int s, t;
    Triple<int32_t> S;
    Triple<T> gv, vec;
    T gd, dist;
};

// The table's sums are double for both types: gfx950's LDS adds 64-bit
// floats at 9 cycles per wave (21 at random addresses) but 32-bit ones at
// 194, one lane after another (measured per CU; 32-bit integers: 5 and 7).
template <typename T>
struct BwdLds {
    alignas(16) int key[kBwdSlots];
    double val[3 * kBwdSlots];
    T acc[kBwdWaves][9];
    int b[kBwdWaves];
    // per wave: atoms and sums that found no slot, in lane order
    T out[kBwdWaves][3 * kWave];
    int out_atom[kBwdWaves][kWave];
};

// The table of a workgroup's pairs: the atoms of the structures of its first
// and last source when they fit (direct), else hashed.
struct BwdTable {
    bool direct;
    int a_lo, span;
};

// The wave's adds to grad_pos of the lanes in `mask`, three lanes per atom.
template <typename T>
__device__ __forceinline__ void add_outside(T* grad_pos, BwdLds<T>& L, int wv, int lane,
                                            unsigned long long mask, int atom, const T (&g)[3]) {
    if (!mask) return;
    wave_lds_fence();
    if ((mask >> lane) & 1ull) {
        const int r = lanes_below(mask);
        L.out_atom[wv][r] = atom;
#pragma unroll
        for (int c = 0; c < 3; ++c) L.out[wv][3 * r + c] = g[c];
    }
    wave_lds_fence();
    const int n = 3 * __popcll(mask);
    for (int i = lane; i < n; i += kWave) {
        const int r = i / 3;
        unsafeAtomicAdd(grad_pos + 3 * (int64_t)L.out_atom[wv][r] + (i - 3 * r), L.out[wv][i]);
    }
}

// Slots of K atoms of the lane in the hashed table, -1 where there is none
// (or where on[k] is false).  A bucket holds four keys, read at once; a
// bucket's slots fill in order and are never freed, so an atom has one slot.
template <typename T, int K>
__device__ __forceinline__ void hash_slots(BwdLds<T>& L, const bool (&on)[K],
                                           const int (&atom)[K], int (&slot)[K]) {
    static_assert((kBwdSlots & (kBwdSlots - 1)) == 0, "a power of two");
    constexpr int kBits = __builtin_ctz(kBwdSlots / 4);
    unsigned h[K];
    bool want[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        h[k] = ((unsigned)atom[k] * 2654435761u) >> (32 - kBits);
        slot[k] = -1;
        want[k] = on[k];
    }
#pragma unroll 1
    for (int p = 0; p < kBwdProbes; ++p) {
        int4 key[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            wave_lds_fence();
            key[k] = *reinterpret_cast<const int4*>(&L.key[4 * h[k]]);
        }
        bool more = false;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (!want[k]) continue;
            const int x = atom[k];
            const int hit = key[k].x == x ? 0 : key[k].y == x ? 1 : key[k].z == x ? 2
                                                    : key[k].w == x ? 3 : -1;
            if (hit >= 0) {
                slot[k] = (int)(4 * h[k]) + hit;
                want[k] = false;
                continue;
            }
            const int free_at = key[k].x == -1 ? 0 : key[k].y == -1 ? 1 : key[k].z == -1 ? 2
                                                    : key[k].w == -1 ? 3 : -1;
            if (free_at >= 0) {
                const int was = atomicCAS(&L.key[4 * h[k] + free_at], -1, x);
                if (was == -1 || was == x) {
                    slot[k] = (int)(4 * h[k]) + free_at;
                    want[k] = false;
                    continue;
                }
                // taken meanwhile: look at the bucket again
            } else {
                h[k] = (h[k] + 1) & (kBwdSlots / 4 - 1);
            }
            more = true;
        }
        if (!__builtin_amdgcn_ballot_w64(more)) break;
    }
}

// The lanes' sums into the table, or into grad_pos.  Every lane calls it.
template <typename T, int K>
__device__ __forceinline__ void table_add(T* grad_pos, BwdLds<T>& L, int wv, int lane,
                                          const bool (&on)[K], const BwdTable& table,
                                          const int (&atom)[K], const T (&g)[K][3]) {
    int slot[K];
    if (table.direct) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            slot[k] = atom[k] - table.a_lo;
            if (!on[k] || (unsigned)slot[k] >= (unsigned)table.span) slot[k] = -1;
        }
    } else {
        hash_slots<T, K>(L, on, atom, slot);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (slot[k] >= 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) atomicAdd(&L.val[3 * slot[k] + c], (double)g[k][c]);
        }
        add_outside(grad_pos, L, wv, lane, ballot(on[k] && slot[k] < 0), atom[k], g[k]);
    }
}

template <typename T>
__device__ __forceinline__ BwdTable open_table(BwdLds<T>& L, int64_t n_atoms, int64_t nb,
                                               const int64_t* bp, int64_t s0, int64_t s1) {
    BwdTable t;
    t.a_lo = 0;
    int64_t span = n_atoms;
    if (nb > 1) {
        const int b0 = uniform(unit_structure(bp, nb, s0));
        const int b1 = uniform(unit_structure(bp, nb, s1));
        t.a_lo = uniform((int)bp[b0]);
        span = bp[b1 + 1] - (int64_t)t.a_lo;
    }
    t.span = uniform(span > 0 && span <= kBwdSlots ? (int)span : 0);
    t.direct = t.span != 0;
    const int tid = threadIdx.x;
    if (t.direct) {
        for (int i = tid; i < 3 * t.span; i += kBwdBlock) L.val[i] = 0.0;
    } else {
        for (int i = tid; i < kBwdSlots; i += kBwdBlock) L.key[i] = -1;
        for (int i = tid; i < 3 * kBwdSlots; i += kBwdBlock) L.val[i] = 0.0;
    }
    __syncthreads();
    return t;
}

// The wave's current structure: its atoms [lo, hi) and per-lane partial sums
// of its cell gradient.
template <typename T>
struct BwdCell {
    T acc[9];
    int b, lo, hi;
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int k = 0; k < 9; ++k) acc[k] = T(0);
    }
    __device__ __forceinline__ void begin() {
        clear();
        b = -1;
        lo = hi = 0;
    }
    __device__ __forceinline__ void add(const Triple<int32_t>& s, const T (&g)[3], bool mine) {
        const T S[3] = {(T)s.x, (T)s.y, (T)s.z};
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int c = 0; c < 3; ++c) acc[3 * a + c] += mine ? S[a] * g[c] : T(0);
    }
    // The structure of atom s becomes the current one; the sums of the last
    // one are added to grad_cell.
    __device__ __forceinline__ void enter(int s, const int64_t* bp, int64_t nb, T* grad_cell) {
        const int lane = lane_id();
        if (b >= 0) {
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                const T x = wave_sum(acc[k]);
                if (lane == kWave - 1) unsafeAtomicAdd(grad_cell + 9 * (int64_t)b + k, x);
            }
            clear();
        }
        // usually one of the next structures: 64 boundaries, one load per lane
        if (b >= 0 && s >= hi) {
            const int64_t at = (int64_t)b + 1 + lane;
            const int64_t v = bp[min(at, nb)];
            const int k = __popcll(ballot(at < nb && v <= (int64_t)s));
            if (k > 0 && k < kWave) {
                lo = __builtin_amdgcn_readlane((int)v, k - 1);
                hi = __builtin_amdgcn_readlane((int)v, k);
                b += k;
                return;
            }
        }
        b = nb == 1 ? 0 : uniform(unit_structure(bp, nb, s));
        lo = uniform((int)bp[b]);
        hi = uniform((int)bp[b + 1]);
    }
};

// Ends a workgroup: the waves' last cell sums, merged where they share a
// structure, and the table's atoms, once each, three lanes per atom.
template <typename T>
__device__ __forceinline__ void close_table(T* grad_pos, T* grad_cell, BwdLds<T>& L, const BwdTable& t,
                                            const BwdCell<T>& cell, int wv, int lane) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const T x = wave_sum(cell.acc[k]);
        if (lane == kWave - 1) L.acc[wv][k] = x;
    }
    if (lane == 0) L.b[wv] = cell.b;
    __syncthreads();
    if (t.direct) {
        for (int i = tid; i < 3 * t.span; i += kBwdBlock) {
            const T v = (T)L.val[i];
            if (v != T(0)) unsafeAtomicAdd(grad_pos + 3 * (int64_t)t.a_lo + i, v);
        }
    } else {
        for (int i = tid; i < 3 * kBwdSlots; i += kBwdBlock) {
            const int slot = i / 3;
            const int key = L.key[slot];
            if (key >= 0)
                unsafeAtomicAdd(grad_pos + 3 * (int64_t)key + (i - 3 * slot), (T)L.val[i]);
        }
    }
    if (tid < 9) {
        for (int w = 0; w < kBwdWaves; ++w) {
            const int bw = L.b[w];
            if (bw < 0) continue;
            bool first = true;
            for (int u = 0; u < w; ++u) first = first && L.b[u] != bw;
            if (!first) continue;
            T sum = T(0);
            for (int u = w; u < kBwdWaves; ++u)
                if (L.b[u] == bw) sum += L.acc[u][tid];
            unsafeAtomicAdd(grad_cell + 9 * (int64_t)bw + tid, sum);
        }
    }
}

// The rows of a list as the backward reads them; GV, GD: the gradients of D
// and of d are given.
template <typename T, bool GV, bool GD>
struct BwdList {
    int64_t n_pairs;
    const int64_t* pairs;
    const int32_t* shifts;
    const T *vec, *dist, *grad_vec, *grad_dist;
    // rows past the list load its last row
    __device__ __forceinline__ BwdRow<T> load(int64_t e) const {
        const int64_t at = min(e, n_pairs - 1);
        BwdRow<T> r;
        const int* st = reinterpret_cast<const int*>(pairs + 2 * at);
        r.s = st[0];
        r.t = st[2];
        r.S = *reinterpret_cast<const Triple<int32_t>*>(shifts + 3 * at);
        if constexpr (GV) r.gv = *reinterpret_cast<const Triple<T>*>(grad_vec + 3 * at);
        if constexpr (GD) {
            r.gd = grad_dist[at];
            r.dist = dist[at];
            r.vec = *reinterpret_cast<const Triple<T>*>(vec + 3 * at);
        }
        return r;
    }
    // dL/dD of a row and its share of dL/dd; 0 where not valid
    __device__ __forceinline__ static void gradient(const BwdRow<T>& r, bool valid, T (&g)[3]) {
        g[0] = g[1] = g[2] = T(0);
        if constexpr (GV) {
            g[0] = r.gv.x;
            g[1] = r.gv.y;
            g[2] = r.gv.z;
        }
        if constexpr (GD) {
            if (r.dist != T(0)) {
                const T q = r.gd / r.dist;
                g[0] += q * r.vec.x;
                g[1] += q * r.vec.y;
                g[2] += q * r.vec.z;
            }
        }
        if (!valid) g[0] = g[1] = g[2] = T(0);
    }
};

// Both gradients cleared in one launch (a second fill cost a small call with
// forces 4 % or more).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_zero_gradients(T* grad_pos, int64_t np, T* grad_cell,
                                                           int64_t nc) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < np)
        grad_pos[i] = T(0);
    else if (i - np < nc)
        grad_cell[i - np] = T(0);
}

// Consecutive pairs: per of them to each wave (backward_pairs_per_wave).
template <typename T, bool GV, bool GD>
__global__ __launch_bounds__(kBwdBlock) void k_geometry_backward(
    BwdList<T, GV, GD> list, int64_t n_atoms, int64_t nb, const int64_t* bp, T* grad_pos,
    T* grad_cell, int64_t per) {
    __shared__ BwdLds<T> L;
    constexpr int K = kBwdRows;
    const int lane = lane_id();
    const int wv = uniform(threadIdx.x / kWave);
    const int64_t n_pairs = list.n_pairs;
    const int64_t b_lo = (int64_t)blockIdx.x * kBwdWaves * per;
    if (b_lo >= n_pairs) return;  // the grid ends at the last pair
    const int64_t b_hi = min(b_lo + kBwdWaves * per, n_pairs);
    const int64_t w_lo = min(b_lo + wv * per, n_pairs);
    const int64_t w_hi = min(w_lo + per, n_pairs);
    BwdRow<T> row[K];
#pragma unroll
    for (int k = 0; k < K; ++k) row[k] = list.load(w_lo + k * kWave + lane);
    int64_t s0 = 0, s1 = 0;
    if (nb > 1) {
        s0 = list.pairs[2 * b_lo];
        s1 = list.pairs[2 * (b_hi - 1)];
    }
    const BwdTable table = open_table(L, n_atoms, nb, bp, s0, s1);
    BwdCell<T> cell;
    cell.begin();
    for (int64_t e0 = w_lo; e0 < w_hi; e0 += K * kWave) {
        BwdRow<T> next[K];
#pragma unroll
        for (int k = 0; k < K; ++k) next[k] = list.load(e0 + (K + k) * kWave + lane);
        bool valid[K], tail[K];
        int s[K], t[K];
        T g[K][3], sum[K][3];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            valid[k] = e0 + k * kWave + lane < w_hi;
            s[k] = valid[k] ? row[k].s : -1;
            t[k] = row[k].t;
            list.gradient(row[k], valid[k], g[k]);
        }
        table_add<T, K>(grad_pos, L, wv, lane, valid, table, t, g);
        // cell side
#pragma unroll
        for (int k = 0; k < K; ++k) {
            unsigned long long left = ballot(valid[k] && (s[k] < cell.lo || s[k] >= cell.hi));
            unsigned long long on = ballot(valid[k]) & ~left;
            for (;;) {
                cell.add(row[k].S, g[k], (on >> lane) & 1ull);
                if (!left) break;
                cell.enter(__builtin_amdgcn_readlane(s[k], __builtin_ctzll(left)), bp, nb,
                           grad_cell);
                // at least the lane that was entered for, whatever bp says
                on = (ballot(s[k] >= cell.lo && s[k] < cell.hi) & left) | (left & (~left + 1ull));
                left &= ~on;
            }
        }
        // source side: runs of equal sources; a run's last lane adds its sum
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int sp = dpp_move<0x138, 0xf>(s[k]);  // wave_shr:1
            const unsigned long long heads = ballot(lane == 0 || sp != s[k]);
            const unsigned long long le = ~0ull >> (kWave - 1 - lane);
            const int seg0 = 63 - __builtin_clzll(heads & le);
            tail[k] = valid[k] && (lane == kWave - 1 || ((heads >> (lane + 1)) & 1ull));
#pragma unroll
            for (int c = 0; c < 3; ++c) sum[k][c] = -g[k][c];
            segment_sums(sum[k], seg0, lane);
        }
        table_add<T, K>(grad_pos, L, wv, lane, tail, table, s, sum);
#pragma unroll
        for (int k = 0; k < K; ++k) row[k] = next[k];
    }
    close_table(grad_pos, grad_cell, L, table, cell, wv, lane);
}

constexpr int kRunMost = 64;  // runs per workgroup, at most

// One source's pairs: rows [first, first + count).
struct SourceRun {
    int64_t first;
    int32_t atom, count;
};

// Runs of each workgroup: about 16,384 pairs (37 M float64 pairs of slabs in
// 94,000 runs: 519 us, 531 at 8,192 pairs, 595 at 4,096; a table of 4,096
// slots with 1,024 threads, one workgroup per CU: 535).
inline int64_t backward_runs_per_block(int64_t n_pairs, int64_t n_runs) {
    const int64_t mean = (n_pairs + n_runs - 1) / n_runs;
    const int64_t r = 16384 / (mean > 0 ? mean : 1);
    return r < 8 ? 8 : r > kRunMost ? kRunMost : r;
}

// The sources of a list in binned order with their rows.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_source_runs(int64_t n, const Vec4<T>* binned,
                                                        const long long* offsets,
                                                        const long long* counts, bool by_bin,
                                                        SourceRun* runs) {
    const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= n) return;
    const int atom = as_idx(binned[k].w);
    const int64_t at = by_bin ? k : atom;
    runs[k] = SourceRun{offsets[at], atom, (int32_t)counts[at]};
}

// The same sums over the sources' runs in an order of their own.  In a list
// in index order consecutive sources lie anywhere in their structure, so the
// table of a workgroup of consecutive pairs overflows (one line request per
// pair outside it); visited in binned order, neighbouring runs share their
// targets.  Each wave takes every eighth run of the workgroup, the next
// rows (of this run or the next one) loading while the current ones are
// summed; a run's source is one wave sum.  37 M float64 pairs of slabs,
// gradient of d: 1.91 ms over consecutive pairs, 519 us over runs (4.8 TB/s;
// streaming the rows takes about 416).
template <typename T, bool GV, bool GD>
__global__ __launch_bounds__(kBwdBlock) void k_geometry_backward_runs(
    BwdList<T, GV, GD> list, const SourceRun* runs, int64_t n_runs, int per, int64_t n_atoms,
    int64_t nb, const int64_t* bp, T* grad_pos, T* grad_cell) {
    __shared__ BwdLds<T> L;
    __shared__ SourceRun s_runs[kRunMost];
    // one pair per lane and round: a second one makes the last round of a
    // run emptier (547 against 531 us)
    constexpr int K = 1;
    const int lane = lane_id();
    const int wv = uniform(threadIdx.x / kWave);
    const int64_t r_lo = (int64_t)blockIdx.x * per;
    if (r_lo >= n_runs) return;  // the grid ends at the last run
    const int n = (int)min((int64_t)per, n_runs - r_lo);
    for (int i = threadIdx.x; i < n; i += kBwdBlock) s_runs[i] = runs[r_lo + i];
    const BwdTable table =
        open_table(L, n_atoms, nb, bp, (int64_t)runs[r_lo].atom, (int64_t)runs[r_lo + n - 1].atom);
    BwdCell<T> cell;
    cell.begin();
    // the wave's position: run r, rows from e on, up to `end`
    int r = wv, atom = 0;
    int64_t e = 0, end = 0;
    auto seek = [&]() {  // the first of the wave's runs from r on that has rows
        for (; r < n; r += kBwdWaves) {
            const SourceRun x = s_runs[r];
            const int count = uniform(x.count);
            if (count <= 0) continue;
            const long long f = (long long)x.first;
            e = max(((int64_t)uniform((int)(f >> 32)) << 32) | (unsigned)uniform((int)f), int64_t{0});
            end = min(e + count, list.n_pairs);
            atom = uniform(x.atom);
            return;
        }
    };
    seek();
    BwdRow<T> row[K];
    if (r < n) {
#pragma unroll
        for (int k = 0; k < K; ++k) row[k] = list.load(e + k * kWave + lane);
    }
    T part[3] = {T(0), T(0), T(0)};  // the lane's share of the run's source
    while (r < n) {
        // the rows in hand
        const int64_t c_e = e, c_end = end;
        const int c_atom = atom;
        // the next ones, of this run or of the wave's next run
        e += K * kWave;
        const bool last = e >= end;
        if (last) {
            r += kBwdWaves;
            seek();
        }
        BwdRow<T> next[K];
#pragma unroll
        for (int k = 0; k < K; ++k) next[k] = list.load((r < n ? e : c_e) + k * kWave + lane);
        if (c_atom < cell.lo || c_atom >= cell.hi) cell.enter(c_atom, bp, nb, grad_cell);
        bool valid[K];
        int t[K];
        T g[K][3];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            valid[k] = c_e + k * kWave + lane < c_end;
            t[k] = row[k].t;
            list.gradient(row[k], valid[k], g[k]);
            cell.add(row[k].S, g[k], valid[k]);
#pragma unroll
            for (int c = 0; c < 3; ++c) part[c] -= g[k][c];
        }
        table_add<T, K>(grad_pos, L, wv, lane, valid, table, t, g);
        if (last) {
            const bool on[1] = {lane == kWave - 1};
            const int a[1] = {c_atom};
            T sum[1][3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                sum[0][c] = wave_sum(part[c]);
                part[c] = T(0);
            }
            table_add<T, 1>(grad_pos, L, wv, lane, on, table, a, sum);
        }
#pragma unroll
        for (int k = 0; k < K; ++k) row[k] = next[k];
    }
    close_table(grad_pos, grad_cell, L, table, cell, wv, lane);
}

}  // namespace tnr
