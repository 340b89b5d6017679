// Shot sampler with qfvm's own rule, evaluated exactly and in parallel.
//
// measure_samples (src/qfvm/statevector.hpp:1380-1412) gives, for each uniform u, the first index k
// whose running sum S_k = fl(S_{k-1} + p_k), p_k = |amp_k|^2, exceeds u (2^n when none does), by
// rescanning the state from index 0 for every shot: O(shots * 2^n). Here S is evaluated once, at
// every 32-element block end, bit for bit equal to that sequential sum, and each shot is a binary
// search over the block ends plus at most 32 sequential additions inside its block.
//
// p_k is what g++ emits for the reference's std::real(d * std::conj(d)) under -O3 -mfma
// -ffast-math: fma(re, re, im * im) in double. The block ends come from integer arithmetic:
// * while S stays in one binade [2^e, 2^(e+1)), S = m 2^(e-52) for an integer m < 2^53 and
//   fl(S + p) = (m + rne(p / 2^(e-52))) 2^(e-52): an integer step of floor(p / ulp), plus one when
//   the fraction is above 1/2; at exactly 1/2 plus one only when that makes m even (ties to even),
//   so the step depends on the parity of the incoming m;
// * a block's effect is therefore a pair (w0, w1), the increment for an even / odd incoming m, and
//   pairs compose associatively: (f then g)_p = f_p + g_{(p + f_p) mod 2};
// * per chunk of blocks (growing geometrically), one kernel forms every block's pair and every
//   tile's pair (64 blocks), one workgroup scans the tiles, one kernel turns the prefixes into m at
//   each block end and reports the first block whose m could reach 2^53 - 1 (the sum may leave the
//   binade there); that block is replayed with double additions from its exact start, and the next
//   chunk starts in the new binade. Blocks before the first nonzero p end at 0.
// Algorithmic bytes of a sample call: about one read of the state (s 2^n) plus 8 bytes per 32
// amplitudes for the block ends, plus shots * (8 + 32 s) for the searches.
#include <algorithm>
#include <climits>
#include <cmath>

#include "common.h"

namespace qfvm {

constexpr int SB = 32;            // amplitudes per block
constexpr int TILE_BLOCKS = 64;   // blocks per tile of the scan (one 256-thread workgroup)
constexpr int64_t XSAT = 1ll << 60;
constexpr int64_t M_CROSS = (1ll << 53) - 1;
constexpr uint64_t NONE = ~0ull;

struct Xfer {
    int64_t w0, w1;  // increment of m for an even / odd incoming m (saturated at XSAT)
};

struct SeqStatus {
    uint64_t first;     // first index with p > 0
    uint64_t crossing;  // first block of the chunk whose m could leave the binade
    uint64_t next;      // first block not yet evaluated
    double s;           // exact S at the end of block next - 1
};

template <typename R>
__device__ __forceinline__ double prob_at(const V2<R>* __restrict__ psi, uint64_t i) {
    const V2<R> a = psi[i];
    const double re = (double)a.x, im = (double)a.y;
    return __fma_rn(re, re, __dmul_rn(im, im));
}

__device__ __forceinline__ Xfer xcompose(Xfer f, Xfer g) {
    Xfer r;
    r.w0 = min(f.w0 + ((f.w0 & 1) ? g.w1 : g.w0), XSAT);
    r.w1 = min(f.w1 + (((f.w1 + 1) & 1) ? g.w1 : g.w0), XSAT);
    return r;
}

// the step of one p in the binade of ulp 2^-sc (lim = the binade's upper end)
__device__ __forceinline__ Xfer xelem(double p, int sc, double lim) {
    if (!(p < lim)) return Xfer{XSAT, XSAT};
    const double r = ldexp(p, sc);  // exact: a power-of-two scaling, r < 2^53
    const double fl = floor(r);
    const double f = r - fl;
    const int64_t q = (int64_t)fl;
    if (f > 0.5) return Xfer{q + 1, q + 1};
    if (f < 0.5) return Xfer{q, q};
    return Xfer{q + (q & 1), q + ((q + 1) & 1)};
}

__global__ void k_seq_init(SeqStatus* st) {
    if (threadIdx.x == 0) {
        st->first = NONE;
        st->crossing = NONE;
        st->next = 0;
        st->s = 0.0;
    }
}

template <typename R>
__global__ void __launch_bounds__(256) k_first_nonzero(const V2<R>* __restrict__ psi, uint64_t size, SeqStatus* st) {
    __shared__ uint64_t wmin[4];
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    uint64_t best = NONE;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < size; i += stride) {
        if (prob_at<R>(psi, i) > 0.0) {
            best = i;
            break;  // later indices of this thread are larger
        }
    }
    // one atomic per workgroup: a dense state would otherwise send every thread to one address
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) best = min(best, (uint64_t)__shfl_xor((unsigned long long)best, o, 64));
    if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        best = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3]));
        if (best != NONE) atomicMin(reinterpret_cast<unsigned long long*>(&st->first), (unsigned long long)best);
    }
}

__device__ __forceinline__ Xfer shfl_down_x(Xfer x, int off) {
    return Xfer{__shfl_down(x.w0, off, 64), __shfl_down(x.w1, off, 64)};
}
__device__ __forceinline__ Xfer shfl_up_x(Xfer x, int off) {
    return Xfer{__shfl_up(x.w0, off, 64), __shfl_up(x.w1, off, 64)};
}

// Inclusive scan over the lanes of a wavefront in lane order (lane i gets lanes 0 .. i composed).
__device__ __forceinline__ Xfer wave_scan_x(Xfer x, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const Xfer o = shfl_up_x(x, off);
        if (lane >= off) x = xcompose(o, x);
    }
    return x;
}

// Composition of the pairs of `width` consecutive lanes in lane order, left in the first lane of each
// run of `width` (a power of two up to 64).
__device__ __forceinline__ Xfer lane_tree_x(Xfer x, int lane, int width) {
    for (int off = 1; off < width; off <<= 1) {
        const Xfer o = shfl_down_x(x, off);
        if ((lane & (2 * off - 1)) == 0) x = xcompose(x, o);
    }
    return x;
}

// Pairs of blocks [blk0, blk0 + nb) (one per block, chunk-relative in bx) and of their tiles (tx).
// The tile's 2048 probabilities are read with contiguous loads (element r 256 + tid per thread and
// row) into LDS; each thread then composes a run of 8 consecutive elements in order, four runs make
// a block (two shuffles) and the tile's 64 blocks are composed in order by wavefront 0 (six).
// Elements past the chunk have p = 0, the identity.
template <typename R>
__global__ void __launch_bounds__(256) k_seq_blocks(const V2<R>* __restrict__ psi, uint64_t blk0, uint64_t nb, int sc,
                                                    double lim, Xfer* __restrict__ bx, Xfer* __restrict__ tx) {
    constexpr int TE = TILE_BLOCKS * SB;  // elements per tile
    constexpr int RUN = 8;                // elements per thread's run
    constexpr int ROWS = TE / 256;
    static_assert(TE == 256 * RUN && SB == 4 * RUN, "one run per thread, four runs per block");
    __shared__ double pl[TE / RUN * (RUN + 1)];  // run-major, padded by one slot per run
    __shared__ Xfer bl[TILE_BLOCKS];
    const int tid = threadIdx.x;
    const uint64_t tb0 = (uint64_t)blockIdx.x * TILE_BLOCKS;  // first block of the tile in the chunk
    const uint64_t ne = min((uint64_t)TILE_BLOCKS, nb - tb0) * SB;
    const V2<R>* __restrict__ src = psi + (blk0 + tb0) * SB;
    double p[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const int e = r * 256 + tid;
        p[r] = (uint64_t)e < ne ? prob_at<R>(src, e) : 0.0;
    }
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const int e = r * 256 + tid;
        pl[(e / RUN) * (RUN + 1) + e % RUN] = p[r];
    }
    __syncthreads();
    Xfer x{0, 0};
#pragma unroll
    for (int j = 0; j < RUN; j++) x = xcompose(x, xelem(pl[tid * (RUN + 1) + j], sc, lim));
    x = lane_tree_x(x, tid & 63, SB / RUN);
    if ((tid & (SB / RUN - 1)) == 0) {
        const int b = tid / (SB / RUN);
        bl[b] = x;
        if (tb0 + b < nb) bx[tb0 + b] = x;
    }
    __syncthreads();
    if (tid < TILE_BLOCKS) {
        const Xfer t = lane_tree_x(bl[tid], tid, TILE_BLOCKS);
        if (tid == 0) tx[blockIdx.x] = t;
    }
}

// Pair of each group of SCAN_GROUP consecutive tiles (one 1024-thread workgroup per group).
constexpr int SCAN_GROUP = 1024;

__global__ void __launch_bounds__(SCAN_GROUP) k_seq_group_sums(const Xfer* __restrict__ tx, uint64_t ntiles,
                                                               Xfer* __restrict__ gx) {
    __shared__ Xfer wt[SCAN_GROUP / 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const uint64_t t = (uint64_t)blockIdx.x * SCAN_GROUP + tid;
    Xfer x = t < ntiles ? tx[t] : Xfer{0, 0};
    x = lane_tree_x(x, lane, 64);
    if (lane == 0) wt[tid >> 6] = x;
    __syncthreads();
    if (tid < SCAN_GROUP / 64) {
        const Xfer g = lane_tree_x(wt[tid], tid, SCAN_GROUP / 64);
        if (tid == 0) gx[blockIdx.x] = g;
    }
}

// Exclusive prefix of every tile of the chunk: the group's prefix (its predecessors' pairs,
// composed by wavefront 0), then an inclusive scan of the group's tiles over shuffles and the 16
// wavefront totals.
__global__ void __launch_bounds__(SCAN_GROUP) k_seq_tile_prefix(const Xfer* __restrict__ tx, uint64_t ntiles,
                                                                const Xfer* __restrict__ gx, Xfer* __restrict__ tpre) {
    __shared__ Xfer wt[SCAN_GROUP / 64];
    __shared__ Xfer gpre;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const uint64_t g = blockIdx.x;
    if (wv == 0) {
        const uint64_t per = (g + 63) / 64;
        const uint64_t a = (uint64_t)lane * per, b = min(a + per, g);
        Xfer x{0, 0};
        for (uint64_t i = a; i < b; i++) x = xcompose(x, gx[i]);
        x = wave_scan_x(x, lane);
        if (lane == 63) gpre = x;
    }
    const uint64_t t = g * SCAN_GROUP + tid;
    const Xfer v = t < ntiles ? tx[t] : Xfer{0, 0};
    const Xfer inc = wave_scan_x(v, lane);
    Xfer ex = shfl_up_x(inc, 1);
    if (lane == 0) ex = Xfer{0, 0};
    if (lane == 63) wt[wv] = inc;
    __syncthreads();
    Xfer pre = gpre;
    for (int j = 0; j < wv; j++) pre = xcompose(pre, wt[j]);
    if (t < ntiles) tpre[t] = xcompose(pre, ex);
}

// m at every block end of the chunk, written to B as the exact double S = m 2^(e-52): one
// wavefront per tile, lane = block, an inclusive scan of the tile's block pairs from the tile's
// prefix. The first block whose m reaches 2^53 - 1 is reported (the atomic keeps the earliest over
// the tiles; a tile that starts at or past it reports its first block) and nothing at or after it
// is written.
__global__ void __launch_bounds__(256) k_seq_apply(const Xfer* __restrict__ bx, const Xfer* __restrict__ tpre,
                                                   uint64_t blk0, uint64_t nb, uint64_t ntiles, int64_t m0, int e52,
                                                   double* __restrict__ B, SeqStatus* st) {
    const int lane = threadIdx.x & 63;
    const uint64_t t = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= ntiles) return;  // whole wavefronts
    const Xfer pre = tpre[t];
    const int64_t mt = m0 + ((m0 & 1) ? pre.w1 : pre.w0);
    const uint64_t cb = t * TILE_BLOCKS + lane;
    const bool in = cb < nb;
    const Xfer inc = wave_scan_x(in ? bx[cb] : Xfer{0, 0}, lane);
    const int64_t m = mt + ((mt & 1) ? inc.w1 : inc.w0);  // nondecreasing over the lanes
    const uint64_t cross = __ballot(in && m >= M_CROSS);
    const int first = cross ? __ffsll((unsigned long long)cross) - 1 : 64;
    // (tiles past a reported crossing skip the atomic: one address would serialise them all)
    if (lane == first && blk0 + cb < *reinterpret_cast<volatile uint64_t*>(&st->crossing))
        atomicMin(reinterpret_cast<unsigned long long*>(&st->crossing), (unsigned long long)(blk0 + cb));
    if (in && lane < first) B[blk0 + cb] = ldexp((double)m, e52);
}

// Closes a chunk: with no crossing, the chunk's last block end is the new start; otherwise (and for
// a block evaluated alone, seq_only) the block is replayed with double additions from its exact
// start. Writes the status the host reads.
template <typename R>
__global__ void k_seq_finish(const V2<R>* __restrict__ psi, uint64_t chunk_start, uint64_t chunk_end, double s_start,
                             int seq_only, int w, double* __restrict__ B, SeqStatus* st) {
    if (threadIdx.x != 0) return;
    const uint64_t c = seq_only ? chunk_start : st->crossing;
    if (c == NONE) {
        st->next = chunk_end;
        st->s = B[chunk_end - 1];
    } else {
        double s = c > chunk_start ? B[c - 1] : s_start;
        for (int k = 0; k < w; k++) s = __dadd_rn(s, prob_at<R>(psi, c * (uint64_t)w + k));
        B[c] = s;
        st->next = c + 1;
        st->s = s;
    }
    st->crossing = NONE;
}

__global__ void __launch_bounds__(256) k_fill_value(double* __restrict__ B, uint64_t a, uint64_t b, double v) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t j = a + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < b; j += stride) B[j] = v;
}

// one shot per thread: first block whose end exceeds u, then the sequential sum inside it
template <typename R>
__global__ void __launch_bounds__(256) k_seq_descend(const V2<R>* __restrict__ psi, const double* __restrict__ B,
                                                     uint64_t nblk, int w, int n, const double* __restrict__ u,
                                                     int64_t shots, uint64_t* __restrict__ out) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= shots) return;
    const double x = u[s];
    if (!(x < B[nblk - 1])) {
        out[s] = 1ull << n;
        return;
    }
    uint64_t lo = 0, hi = nblk - 1;  // B[hi] > x
    while (lo < hi) {
        const uint64_t mid = lo + (hi - lo) / 2;
        if (B[mid] > x)
            hi = mid;
        else
            lo = mid + 1;
    }
    double acc = lo > 0 ? B[lo - 1] : 0.0;
    const uint64_t base = lo * (uint64_t)w;
    uint64_t res = base + (uint64_t)w - 1;
    for (int k = 0; k < w; k++) {
        acc = __dadd_rn(acc, prob_at<R>(psi, base + k));
        if (x < acc) {
            res = base + k;
            break;
        }
    }
    out[s] = res;
}

// ------------------------------------------------------------------------------------------------
// States of up to 4 GiB: every block end without a host round trip per binade.
// The chunk loop above learns where S leaves a binade by reaching it, and waits for the host there: some
// 25 times for 26 qubits. Here a first read sums the probabilities in any order. Such a sum A of the
// blocks before b and the sequential S differ by their roundings, some sqrt(N) 2^-53 of S if these do not
// conspire, so with a margin eps of 32 times that it tells the binade of every block but those whose
// interval [A_b (1 - eps), A_b+1 (1 + eps)] holds a power of two. A second read forms the pairs of the former
// (for their own binade) and marks the latter special: they are replayed with double additions, by one
// thread, in order, each from the end of the one before and the composed pairs between. Blocks that cannot
// change S (all p zero, or below half an ulp of both binades of the interval) are the identity and not
// special. Exactness does not rest on the margin: every pair's use is checked against the exact S (its
// binade, no carry out of it). A block that cannot change S needs no such check: its 32 terms are each
// below 2^-53 of the lower of its two binades, so it can hold only one of their ends, and S is in
// one of the two unless it is off by a factor of nearly two, where N 2^-53 bounds it. A check that fails,
// more than SEQ_SPECIALS special blocks, or sums that are not finite hand over to the chunk loop, which
// goes on from the first block concerned: the ends before it are exact. (A tail of equal terms drifts
// from A beyond the margin, all roundings being the same. One amplitude of probability 1 - 10^-k and such a
// tail, k = 5 to 11: 24 qubits at most 0.43 ms, 26 at most 1.02, 27 at most 1.86, where starting over
// took up to 1.03, 1.57 and 2.31 ms and the chunk loop alone takes 0.87, 1.13 and 1.53. A special block costs 0.4
// us, so more than 256 of them are better left to the loop: k = 9 at 24 qubits 0.70 -> 0.43 ms.)
// What bounds it: two reads of the state, and some 40 us of launches up to 18 qubits; the chunk loop
// reads once, so it stays the better one for larger states, whose reads outweigh its waits (SEQ_BYTES:
// 28 qubits at complex128 1.84 -> 1.63 ms; two reads of 29 qubits would take 3.2, one and the waits 2.7).
// Measured for one shot of a random complex128 state: 12 qubits 268 -> 48 us, 18 qubits 469 -> 52 us, 24
// qubits 818 -> 151 us, 26 qubits 1.11 -> 0.45 ms.
constexpr uint64_t SEQ_BYTES = 4ull << 30;
constexpr unsigned SEQ_SPECIALS = 256;
constexpr int SEQ_IDENTITY = -32768;  // exponent entry of a block that keeps S
constexpr double SEQ_TINY = 0x1p-1000;  // below it every block that changes S is special

struct SegX {      // composed pairs since the last special block, and the number of special blocks
    Xfer x;
    unsigned count;
};
struct SeqSpecial {
    uint64_t block;
    Xfer before;  // pairs between the special block before and this one
};
struct SeqFast {
    uint64_t bad;    // first block whose end is not known to be exact (NONE: all are)
    uint64_t total;  // special blocks
};

__device__ __forceinline__ SegX seg_compose(SegX f, SegX g) {
    return SegX{g.count ? g.x : xcompose(f.x, g.x), f.count + g.count};
}
__device__ __forceinline__ SegX shfl_up_seg(SegX v, int off) {
    return SegX{shfl_up_x(v.x, off), (unsigned)__shfl_up((int)v.count, off, 64)};
}
__device__ __forceinline__ SegX wave_scan_seg(SegX v, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const SegX o = shfl_up_seg(v, off);
        if (lane >= off) v = seg_compose(o, v);
    }
    return v;
}

// sum of every tile's probabilities
template <typename R>
__global__ void __launch_bounds__(256) k_seq_mass(const V2<R>* __restrict__ psi, uint64_t size, double* __restrict__ mass,
                                                  SeqFast* st) {
    constexpr int TE = TILE_BLOCKS * SB;
    __shared__ double wsum[4];
    const int tid = threadIdx.x;
    if (blockIdx.x == 0 && tid == 0) *st = SeqFast{NONE, 0};
    const uint64_t at = (uint64_t)blockIdx.x * TE;
    double a = 0.0;
#pragma unroll
    for (int r = 0; r < TE / 256; r++)
        if (at + r * 256 + tid < size) a += prob_at<R>(psi, at + r * 256 + tid);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
    if ((tid & 63) == 0) wsum[tid >> 6] = a;
    __syncthreads();
    if (tid == 0) mass[blockIdx.x] = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
}

// exclusive prefix sums of the tiles' masses; each workgroup of SCAN_GROUP tiles adds up those before its own
__global__ void __launch_bounds__(SCAN_GROUP) k_seq_mass_prefix(const double* __restrict__ mass, uint64_t ntiles,
                                                                double* __restrict__ pre) {
    __shared__ double wtot[SCAN_GROUP / 64], wbefore[SCAN_GROUP / 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const uint64_t first = (uint64_t)blockIdx.x * SCAN_GROUP;
    double before = 0.0;
#pragma unroll 8
    for (uint64_t t = tid; t < first; t += SCAN_GROUP) before += mass[t];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    const double m = first + tid < ntiles ? mass[first + tid] : 0.0;
    double inc = m;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double o = __shfl_up(inc, off, 64);
        if (lane >= off) inc += o;
    }
    double ex = __shfl_up(inc, 1, 64);
    if (lane == 0) {
        ex = 0.0;
        wbefore[wv] = before;
    }
    if (lane == 63) wtot[wv] = inc;
    __syncthreads();
    for (int j = 0; j < SCAN_GROUP / 64; j++) ex += wbefore[j] + (j < wv ? wtot[j] : 0.0);
    if (first + tid < ntiles) pre[first + tid] = ex;
}

// reports the first of a wavefront's blocks (ascending over its lanes) that is not good
__device__ __forceinline__ void seq_report(bool good, uint64_t block, SeqFast* st) {
    const uint64_t m = __ballot(!good);
    // (blocks past a reported one skip the atomic: one address would serialise them all)
    if (m && (int)(threadIdx.x & 63) == __ffsll((unsigned long long)m) - 1 &&
        block < *reinterpret_cast<volatile uint64_t*>(&st->bad))
        atomicMin(reinterpret_cast<unsigned long long*>(&st->bad), (unsigned long long)block);
}

// Pairs of every block for its binade (bx, its exponent in be), the tile's special blocks (mask) and its
// composition (tx). Threads as in k_seq_blocks.
template <typename R>
__global__ void __launch_bounds__(256) k_seq_pairs(const V2<R>* __restrict__ psi, uint64_t nblk,
                                                   const double* __restrict__ pre, double eps, Xfer* __restrict__ bx,
                                                   int16_t* __restrict__ be, uint64_t* __restrict__ mask,
                                                   Xfer* __restrict__ tx, SeqFast* st) {
    constexpr int TE = TILE_BLOCKS * SB, RUN = 8, ROWS = TE / 256;
    __shared__ double pl[TE / RUN * (RUN + 1)];
    __shared__ Xfer bl[TILE_BLOCKS];
    __shared__ double wtot[4];
    __shared__ uint64_t wmask[4];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    // (last tile first: the sums' read leaves the end of the state in the last-level cache)
    const uint64_t tile = gridDim.x - 1 - blockIdx.x, tb0 = tile * TILE_BLOCKS;
    const uint64_t ne = min((uint64_t)TILE_BLOCKS, nblk - tb0) * SB;
    const V2<R>* __restrict__ src = psi + tb0 * SB;
    {
        double p[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const int e = r * 256 + tid;
            p[r] = (uint64_t)e < ne ? prob_at<R>(src, e) : 0.0;
        }
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const int e = r * 256 + tid;
            pl[(e / RUN) * (RUN + 1) + e % RUN] = p[r];
        }
    }
    __syncthreads();
    double p[RUN], q = 0.0, most = 0.0;
#pragma unroll
    for (int j = 0; j < RUN; j++) {
        p[j] = pl[tid * (RUN + 1) + j];
        q += p[j];
        most = fmax(most, p[j]);
    }
#pragma unroll
    for (int o = 1; o < SB / RUN; o <<= 1) {  // over the block's four threads
        q += __shfl_xor(q, o, 64);
        most = fmax(most, __shfl_xor(most, o, 64));
    }
    double inc = q;  // over the wavefront's 16 blocks
#pragma unroll
    for (int off = SB / RUN; off < 64; off <<= 1) {
        const double o = __shfl_up(inc, off, 64);
        if (lane >= off) inc += o;
    }
    if (lane == 63) wtot[wv] = inc;
    __syncthreads();
    double a0 = pre[tile] + (inc - q);
    for (int j = 0; j < wv; j++) a0 += wtot[j];
    const double a1 = a0 + q;
    const double lo = a0 * (1.0 - eps), hi = a1 * (1.0 + eps);
    bool special = false;
    int e = SEQ_IDENTITY;
    const bool finite = a1 <= 1.7976931348623157e308;
    seq_report(finite, tb0 + tid / (SB / RUN), st);
    if (finite && q > 0.0) {
        if (lo < SEQ_TINY) {
            special = true;
        } else {
            e = ilogb(lo);
            const int eh = ilogb(hi);
            if (eh > e) {
                special = eh > e + 1 || !(most < ldexp(1.0, e - 53));
                e = SEQ_IDENTITY;
            }
        }
    }
    // Without a tie the pair's entries are equal, the sum of the rounded steps: whole numbers below 2^53 (the
    // block ends below its binade's top), exact in double.
    Xfer x{0, 0};
    double sum = 0.0;
    bool tie = false;
    if (e != SEQ_IDENTITY) {
#pragma unroll
        for (int j = 0; j < RUN; j++) {
            const double f = ldexp(p[j], 52 - e), w = rint(f);
            tie = tie || fabs(f - w) == 0.5;
            sum += w;
        }
    }
    if (__any(tie)) {
        if (e != SEQ_IDENTITY) {
            const double lim = ldexp(1.0, e + 1);
            for (int j = 0; j < RUN; j++) x = xcompose(x, xelem(pl[tid * (RUN + 1) + j], 52 - e, lim));
        }
        x = lane_tree_x(x, lane, SB / RUN);
    } else {
#pragma unroll
        for (int o = 1; o < SB / RUN; o <<= 1) sum += __shfl_xor(sum, o, 64);
        x.w0 = x.w1 = (int64_t)sum;
    }
    uint64_t marks = __ballot(special && (lane & (SB / RUN - 1)) == 0);  // bits 0, 4, 8, ...: to bits 0, 1, 2, ...
    if ((tid & (SB / RUN - 1)) == 0) {
        const int b = tid / (SB / RUN);
        bl[b] = x;
        if (tb0 + b < nblk) {
            bx[tb0 + b] = x;
            be[tb0 + b] = (int16_t)e;
        }
    }
    if (lane == 0) {
        uint64_t m = 0;
        for (int b = 0; b < 16; b++) m |= ((marks >> (4 * b)) & 1ull) << b;
        wmask[wv] = m;
    }
    __syncthreads();
    if (tid < TILE_BLOCKS) {
        const uint64_t m = wmask[0] | (wmask[1] << 16) | (wmask[2] << 32) | (wmask[3] << 48);
        // pairs after the last special block (all, if there is none)
        const bool counts = m == 0 || tid > 63 - __clzll((long long)m);
        const Xfer t = lane_tree_x(counts ? bl[tid] : Xfer{0, 0}, tid, TILE_BLOCKS);
        if (tid == 0) {
            tx[tile] = t;
            mask[tile] = m;
        }
    }
}

__device__ __forceinline__ SegX seg_tile(const Xfer* __restrict__ tx, const uint64_t* __restrict__ mask, uint64_t t,
                                         uint64_t ntiles) {
    return t < ntiles ? SegX{tx[t], (unsigned)__popcll(mask[t])} : SegX{Xfer{0, 0}, 0};
}

// composition of each group of SCAN_GROUP consecutive tiles
__global__ void __launch_bounds__(SCAN_GROUP) k_seg_group_sums(const Xfer* __restrict__ tx,
                                                               const uint64_t* __restrict__ mask, uint64_t ntiles,
                                                               SegX* __restrict__ gx) {
    __shared__ SegX wt[SCAN_GROUP / 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const SegX v = wave_scan_seg(seg_tile(tx, mask, (uint64_t)blockIdx.x * SCAN_GROUP + tid, ntiles), lane);
    if (lane == 63) wt[tid >> 6] = v;
    __syncthreads();
    if (tid == 0) {
        SegX g = wt[0];
        for (int j = 1; j < SCAN_GROUP / 64; j++) g = seg_compose(g, wt[j]);
        gx[blockIdx.x] = g;
    }
}

// exclusive prefix of every tile (as k_seq_tile_prefix); the last one's inclusive count is the total
__global__ void __launch_bounds__(SCAN_GROUP) k_seg_tile_prefix(const Xfer* __restrict__ tx,
                                                                const uint64_t* __restrict__ mask, uint64_t ntiles,
                                                                const SegX* __restrict__ gx, SegX* __restrict__ tpre,
                                                                SeqFast* st) {
    __shared__ SegX wt[SCAN_GROUP / 64];
    __shared__ SegX gpre;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const uint64_t g = blockIdx.x;
    if (wv == 0) {
        const uint64_t per = (g + 63) / 64;
        const uint64_t a = (uint64_t)lane * per, b = min(a + per, g);
        SegX x{Xfer{0, 0}, 0};
        for (uint64_t i = a; i < b; i++) x = seg_compose(x, gx[i]);
        x = wave_scan_seg(x, lane);
        if (lane == 63) gpre = x;
    }
    const uint64_t t = g * SCAN_GROUP + tid;
    const SegX inc = wave_scan_seg(seg_tile(tx, mask, t, ntiles), lane);
    SegX ex = shfl_up_seg(inc, 1);
    if (lane == 0) ex = SegX{Xfer{0, 0}, 0};
    if (lane == 63) wt[wv] = inc;
    __syncthreads();
    SegX pre = gpre;
    for (int j = 0; j < wv; j++) pre = seg_compose(pre, wt[j]);
    if (t < ntiles) tpre[t] = seg_compose(pre, ex);
    if (t == ntiles - 1) st->total = pre.count + inc.count;
}

// block `lane` of tile t: the pairs since the last special block, its own included (identity for a special one)
__device__ __forceinline__ Xfer seg_block(const Xfer* __restrict__ bx, const SegX& pre, uint64_t m, uint64_t t, int lane,
                                          uint64_t nblk) {
    const uint64_t cb = t * TILE_BLOCKS + lane;
    const SegX v{cb < nblk ? bx[cb] : Xfer{0, 0}, (unsigned)((m >> lane) & 1ull)};
    const SegX inc = wave_scan_seg(v, lane);
    return inc.count ? inc.x : xcompose(pre.x, inc.x);
}

// the special blocks in order, one wavefront per tile
__global__ void __launch_bounds__(256) k_seq_specials(const Xfer* __restrict__ bx, const uint64_t* __restrict__ mask,
                                                      const SegX* __restrict__ tpre, uint64_t ntiles, uint64_t nblk,
                                                      SeqSpecial* __restrict__ sp) {
    const int lane = threadIdx.x & 63;
    const uint64_t t = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= ntiles) return;  // whole wavefronts
    const uint64_t m = mask[t];
    if (m == 0) return;
    const SegX pre = tpre[t];
    const Xfer x = seg_block(bx, pre, m, t, lane, nblk);
    Xfer before = shfl_up_x(x, 1);
    if (lane == 0) before = pre.x;
    const unsigned k = pre.count + (unsigned)__popcll(m & ((1ull << lane) - 1));
    if (((m >> lane) & 1ull) && k < SEQ_SPECIALS) sp[k] = SeqSpecial{t * TILE_BLOCKS + lane, before};
}

// m 2^(e-52) for the S that the pairs x make of s (s itself where they change nothing)
__device__ __forceinline__ double seq_after(double s, Xfer x, int* e, int64_t* m) {
    *e = ilogb(s);
    const int64_t m0 = (int64_t)ldexp(s, 52 - *e);
    const int64_t w = (m0 & 1) ? x.w1 : x.w0;
    *m = m0 + w;
    return w ? ldexp((double)*m, *e - 52) : s;
}

// S at the end of every special block: their probabilities are staged in LDS, then one thread adds in order
template <typename R>
__global__ void __launch_bounds__(256) k_seq_resolve(const V2<R>* __restrict__ psi, const SeqSpecial* __restrict__ sp,
                                                     double* __restrict__ ends, SeqFast* st) {
    constexpr int BATCH = 128;
    __shared__ double p[BATCH * SB];
    __shared__ Xfer before[BATCH];
    const unsigned total = (unsigned)min(st->total, (uint64_t)SEQ_SPECIALS);
    double s = 0.0;
    for (unsigned k0 = 0; k0 < total; k0 += BATCH) {
        const unsigned n = min((unsigned)BATCH, total - k0);
        __syncthreads();
        for (unsigned i = threadIdx.x; i < n * SB; i += 256) p[i] = prob_at<R>(psi, sp[k0 + i / SB].block * SB + i % SB);
        for (unsigned i = threadIdx.x; i < n; i += 256) before[i] = sp[k0 + i].before;
        __syncthreads();
        if (threadIdx.x == 0)
            for (unsigned k = 0; k < n; k++) {
                int e;
                int64_t m;
                if (s > 0.0) s = seq_after(s, before[k], &e, &m);
#pragma unroll
                for (int j = 0; j < SB; j++) s = __dadd_rn(s, p[k * SB + j]);
                ends[k0 + k] = s;
            }
    }
}

// S at every block end, and the check of every pair's binade
__global__ void __launch_bounds__(256) k_seq_ends(const Xfer* __restrict__ bx, const int16_t* __restrict__ be,
                                                  const uint64_t* __restrict__ mask, const SegX* __restrict__ tpre,
                                                  uint64_t ntiles, uint64_t nblk, const double* __restrict__ ends,
                                                  double* __restrict__ B, SeqFast* st) {
    const int lane = threadIdx.x & 63;
    const uint64_t t = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= ntiles) return;  // whole wavefronts
    const uint64_t m = mask[t];
    const SegX pre = tpre[t];
    const Xfer x = seg_block(bx, pre, m, t, lane, nblk);
    const uint64_t cb = t * TILE_BLOCKS + lane;
    const bool in = cb < nblk;
    const unsigned k = pre.count + (unsigned)__popcll(m & ((2ull << lane) - 1));  // special blocks up to this one
    const bool known = k <= SEQ_SPECIALS;
    const double s = k > 0 && known ? ends[k - 1] : 0.0;
    const int want = in ? be[cb] : SEQ_IDENTITY;
    double end = s;
    bool good = known && s <= 1.7976931348623157e308;
    if (s > 0.0 && good) {
        int e;
        int64_t mm;
        end = seq_after(s, x, &e, &mm);
        if (want != SEQ_IDENTITY) good = want == e && mm < M_CROSS;
    } else if (want != SEQ_IDENTITY) {
        good = false;
    }
    seq_report(good || !in, cb, st);
    if (in) B[cb] = end;
}

// scratch of the chunk loop (sample_typed); the block ends come first, as in sample_fast
struct SeqScratch {
    size_t b, bx, tx, gx, st, u, o;
    uint64_t chunk_max;
    SeqScratch(uint64_t nblk, int64_t shots) {
        auto align = [](size_t x) { return (x + 255) & ~size_t(255); };
        chunk_max = std::min<uint64_t>(nblk, 1ull << 24);
        const uint64_t tiles_max = (chunk_max + TILE_BLOCKS - 1) / TILE_BLOCKS;
        const uint64_t groups_max = (tiles_max + SCAN_GROUP - 1) / SCAN_GROUP;
        b = align(nblk * sizeof(double));
        bx = align(chunk_max * sizeof(Xfer));
        tx = align(tiles_max * sizeof(Xfer));
        gx = align(groups_max * sizeof(Xfer));
        st = align(sizeof(SeqStatus));
        u = align((size_t)shots * sizeof(double));
        o = align((size_t)shots * sizeof(uint64_t));
    }
    size_t bytes() const { return b + bx + 2 * tx + gx + st + u + o; }
};

// Block ends and shots of a state of up to SEQ_BYTES. Returns the first block whose end could not be
// told (NONE: all were, and host_out is written); the ends before it are at the start of the scratch
// and *last is the last of them.
template <typename R>
static uint64_t sample_fast(State& s, const double* host_u, int64_t shots, uint64_t* host_out, double* last) {
    const uint64_t nblk = s.size / SB;
    const uint64_t ntiles = (nblk + TILE_BLOCKS - 1) / TILE_BLOCKS;
    const uint64_t ngroups = (ntiles + SCAN_GROUP - 1) / SCAN_GROUP;
    size_t bytes = 0;
    auto part = [&](size_t b) {
        const size_t at = bytes;
        bytes += (b + 255) & ~size_t(255);
        return at;
    };
    const size_t oB = part(nblk * sizeof(double)), obx = part(nblk * sizeof(Xfer)), obe = part(nblk * sizeof(int16_t));
    const size_t omass = part(ntiles * sizeof(double)), opre = part(ntiles * sizeof(double)), omask = part(ntiles * sizeof(uint64_t));
    const size_t otx = part(ntiles * sizeof(Xfer)), otpre = part(ntiles * sizeof(SegX)), ogx = part(ngroups * sizeof(SegX));
    const size_t osp = part(SEQ_SPECIALS * sizeof(SeqSpecial)), oends = part(SEQ_SPECIALS * sizeof(double));
    const size_t ost = part(sizeof(SeqFast));
    // Up to 2^20 shots: uniforms and results stay in pinned memory, which the search reads and writes; the host
    // copies the uniforms there while the scan runs. 26 qubits: 100000 shots 533 -> 494 us, 200000 shots 651 -> 583.
    const bool few = shots <= (1 << 20);
    const size_t ou = part(few ? 0 : (size_t)shots * sizeof(double)), oo = part(few ? 0 : (size_t)shots * sizeof(uint64_t));
    // (the chunk loop may go on with it, and a larger scratch would lose the ends)
    char* base = reinterpret_cast<char*>(s.ensure_scratch(std::max(bytes, SeqScratch(nblk, shots).bytes())));
    const size_t per = few ? (size_t)shots : 0;
    double* pin = s.ensure_pinned(sizeof(SeqFast) + per * (sizeof(double) + sizeof(uint64_t)));
    SeqFast* hst = reinterpret_cast<SeqFast*>(pin);
    static_assert(sizeof(SeqFast) == 2 * sizeof(double), "pinned layout");
    double* hu = pin + 2;
    uint64_t* ho = reinterpret_cast<uint64_t*>(hu + per);
    auto at = [&](size_t o) { return base + o; };
    double* B = reinterpret_cast<double*>(at(oB));
    Xfer *bx = reinterpret_cast<Xfer*>(at(obx)), *tx = reinterpret_cast<Xfer*>(at(otx));
    int16_t* be = reinterpret_cast<int16_t*>(at(obe));
    double *mass = reinterpret_cast<double*>(at(omass)), *pre = reinterpret_cast<double*>(at(opre)), *ends = reinterpret_cast<double*>(at(oends));
    uint64_t* mask = reinterpret_cast<uint64_t*>(at(omask));
    SegX *tpre = reinterpret_cast<SegX*>(at(otpre)), *gx = reinterpret_cast<SegX*>(at(ogx));
    SeqSpecial* sp = reinterpret_cast<SeqSpecial*>(at(osp));
    SeqFast* st = reinterpret_cast<SeqFast*>(at(ost));
    double* du = few ? hu : reinterpret_cast<double*>(at(ou));
    uint64_t* dout = few ? ho : reinterpret_cast<uint64_t*>(at(oo));
    const V2<R>* psi = reinterpret_cast<const V2<R>*>(s.psi);
    const double eps = (32.0 * std::sqrt((double)s.size) + 1024.0) * 0x1p-53;
    const dim3 tiles((unsigned)ntiles), waves((unsigned)((ntiles + 3) / 4)), groups((unsigned)ngroups);
    if (!few)
        QFVM_HIP(hipMemcpyAsync(du, host_u, (size_t)shots * sizeof(double), hipMemcpyHostToDevice, s.stream));
    {
        KernelScope ks(s, "sample_scan", 2.0 * (double)s.size * s.amp_bytes() + (double)nblk * sizeof(double));
        hipLaunchKernelGGL(k_seq_mass<R>, tiles, dim3(256), 0, s.stream, psi, s.size, mass, st);
        QFVM_LAUNCHED();
        hipLaunchKernelGGL(k_seq_mass_prefix, groups, dim3(SCAN_GROUP), 0, s.stream, mass, ntiles, pre);
        QFVM_LAUNCHED();
        hipLaunchKernelGGL(k_seq_pairs<R>, tiles, dim3(256), 0, s.stream, psi, nblk, pre, eps, bx, be, mask, tx, st);
        QFVM_LAUNCHED();
        if (ngroups > 1) {
            hipLaunchKernelGGL(k_seg_group_sums, groups, dim3(SCAN_GROUP), 0, s.stream, tx, mask, ntiles, gx);
            QFVM_LAUNCHED();
        }
        hipLaunchKernelGGL(k_seg_tile_prefix, groups, dim3(SCAN_GROUP), 0, s.stream, tx, mask, ntiles, gx, tpre, st);
        QFVM_LAUNCHED();
        hipLaunchKernelGGL(k_seq_specials, waves, dim3(256), 0, s.stream, bx, mask, tpre, ntiles, nblk, sp);
        QFVM_LAUNCHED();
        hipLaunchKernelGGL(k_seq_resolve<R>, dim3(1), dim3(256), 0, s.stream, psi, sp, ends, st);
        QFVM_LAUNCHED();
        hipLaunchKernelGGL(k_seq_ends, waves, dim3(256), 0, s.stream, bx, be, mask, tpre, ntiles, nblk, ends, B, st);
        QFVM_LAUNCHED();
    }
    if (few) std::copy(host_u, host_u + shots, hu);
    {
        KernelScope ks(s, "sample_search", (double)shots * (8.0 + SB * (double)s.amp_bytes()));
        hipLaunchKernelGGL(k_seq_descend<R>, dim3((unsigned)((shots + 255) / 256)), dim3(256), 0, s.stream, psi, B, nblk,
                           SB, s.n, du, shots, dout);
        QFVM_LAUNCHED();
    }
    QFVM_HIP(hipMemcpyAsync(hst, st, sizeof(SeqFast), hipMemcpyDeviceToHost, s.stream));
    QFVM_HIP(hipStreamSynchronize(s.stream));
    if (hst->bad != NONE) {
        const uint64_t bad = hst->bad;
        *last = 0.0;
        if (bad > 0) {
            QFVM_HIP(hipMemcpyAsync(pin, B + bad - 1, sizeof(double), hipMemcpyDeviceToHost, s.stream));
            QFVM_HIP(hipStreamSynchronize(s.stream));
            *last = *pin;
        }
        return bad;
    }
    if (few)
        std::copy(ho, ho + shots, host_out);
    else {
        QFVM_HIP(hipMemcpyAsync(host_out, dout, (size_t)shots * sizeof(uint64_t), hipMemcpyDeviceToHost, s.stream));
        QFVM_HIP(hipStreamSynchronize(s.stream));
    }
    return NONE;
}

// from > 0: the ends of the blocks before it are at hand (sample_fast), S = `at` at the last of them
template <typename R>
static void sample_typed(State& s, const double* host_u, int64_t shots, uint64_t* host_out, uint64_t from = 0,
                         double at = 0.0) {
    const int n = s.n;
    const uint64_t size = s.size;
    const int w = size >= (uint64_t)SB ? SB : (int)size;
    const uint64_t nblk = size / (uint64_t)w;
    const SeqScratch sz(nblk, shots);
    const uint64_t chunk_max = sz.chunk_max;
    char* base = reinterpret_cast<char*>(s.ensure_scratch(sz.bytes()));
    double* B = reinterpret_cast<double*>(base);
    Xfer* bx = reinterpret_cast<Xfer*>(base + sz.b);
    Xfer* tx = reinterpret_cast<Xfer*>(base + sz.b + sz.bx);
    Xfer* tpre = reinterpret_cast<Xfer*>(base + sz.b + sz.bx + sz.tx);
    Xfer* gx = reinterpret_cast<Xfer*>(base + sz.b + sz.bx + 2 * sz.tx);
    char* tail = base + sz.b + sz.bx + 2 * sz.tx + sz.gx;
    SeqStatus* st = reinterpret_cast<SeqStatus*>(tail);
    double* du = reinterpret_cast<double*>(tail + sz.st);
    uint64_t* dout = reinterpret_cast<uint64_t*>(tail + sz.st + sz.u);
    SeqStatus* hst = reinterpret_cast<SeqStatus*>(s.ensure_pinned(sizeof(SeqStatus)));
    const V2<R>* psi = reinterpret_cast<const V2<R>*>(s.psi);
    auto read_status = [&] {
        QFVM_HIP(hipMemcpyAsync(hst, st, sizeof(SeqStatus), hipMemcpyDeviceToHost, s.stream));
        QFVM_HIP(hipStreamSynchronize(s.stream));
    };

    {
        KernelScope ks(s, "sample_scan", (double)size * s.amp_bytes() + (double)nblk * sizeof(double));
        hipLaunchKernelGGL(k_seq_init, dim3(1), dim3(64), 0, s.stream, st);
        QFVM_LAUNCHED();
        uint64_t b0 = 0;
        uint64_t next = nblk;
        double S = 0.0;
        if (from > 0) {
            next = from;
            S = at;
        } else {
            hipLaunchKernelGGL(k_first_nonzero<R>, dim3(grid_for(size, 256, 2048)), dim3(256), 0, s.stream, psi, size,
                               st);
            QFVM_LAUNCHED();
            read_status();
            b0 = hst->first == NONE ? nblk : hst->first / (uint64_t)w;
            if (b0 > 0) launch_zero(s, B, b0 * sizeof(double));
        }
        double rate = 0.0;  // growth of S per block over the last evaluated span
        auto finish = [&](uint64_t start, uint64_t end, double s_start, int seq_only) {
            hipLaunchKernelGGL(k_seq_finish<R>, dim3(1), dim3(64), 0, s.stream, psi, start, end, s_start, seq_only, w, B,
                               st);
            QFVM_LAUNCHED();
            read_status();
            next = hst->next;
            S = hst->s;
            rate = next > start ? (S - s_start) / (double)(next - start) : 0.0;
        };
        int singles = 0;  // consecutive blocks replayed alone because a crossing was expected there
        if (from == 0 && b0 < nblk) finish(b0, b0 + 1, 0.0, 1);
        const uint64_t min_chunk = 1ull << 12;
        while (next < nblk) {
            if (!std::isfinite(S)) {  // inf / NaN amplitudes: the sum stays where it is
                hipLaunchKernelGGL(k_fill_value, dim3(grid_for(nblk - next, 256)), dim3(256), 0, s.stream, B, next, nblk,
                                   S);
                QFVM_LAUNCHED();
                break;
            }
            if (!(S >= 2.2250738585072014e-308)) {  // subnormal start: one block at a time
                finish(next, next + 1, S, 1);
                continue;
            }
            const int e = std::ilogb(S);
            const int64_t m0 = (int64_t)std::ldexp(S, 52 - e);
            uint64_t len = std::min(std::max(min_chunk, next - b0), chunk_max);
            if (rate > 0.0 && std::isfinite(rate)) {
                // Blocks until S reaches its binade's top at the last span's rate (performance only:
                // any chunk gives exact results). A crossing expected in the first block is one
                // replayed block, not a chunk read in vain; a crossing expected well before the
                // chunk's end ends the chunk shortly after it.
                const double need = (std::ldexp(1.0, e + 1) - S) / rate;
                if (need < 1.0 && singles < 4) {
                    singles++;
                    finish(next, next + 1, S, 1);
                    continue;
                }
                const double cap = need * 1.25 + (double)TILE_BLOCKS;
                if (cap < (double)len) len = std::max<uint64_t>((uint64_t)cap, 1);
            }
            singles = 0;
            const uint64_t end = std::min(nblk, next + len);
            const uint64_t nb = end - next;
            const uint64_t ntiles = (nb + TILE_BLOCKS - 1) / TILE_BLOCKS;
            hipLaunchKernelGGL(k_seq_blocks<R>, dim3((unsigned)ntiles), dim3(256), 0, s.stream, psi, next, nb, 52 - e,
                               std::ldexp(1.0, e + 1), bx, tx);
            QFVM_LAUNCHED();
            const uint64_t ngroups = (ntiles + SCAN_GROUP - 1) / SCAN_GROUP;
            hipLaunchKernelGGL(k_seq_group_sums, dim3((unsigned)ngroups), dim3(SCAN_GROUP), 0, s.stream, tx, ntiles, gx);
            QFVM_LAUNCHED();
            hipLaunchKernelGGL(k_seq_tile_prefix, dim3((unsigned)ngroups), dim3(SCAN_GROUP), 0, s.stream, tx, ntiles, gx,
                               tpre);
            QFVM_LAUNCHED();
            hipLaunchKernelGGL(k_seq_apply, dim3((unsigned)((ntiles + 3) / 4)), dim3(256), 0, s.stream, bx, tpre, next,
                               nb, ntiles, m0, e - 52, B, st);
            QFVM_LAUNCHED();
            finish(next, end, S, 0);
        }
    }
    if (shots <= 0) return;
    QFVM_HIP(hipMemcpyAsync(du, host_u, (size_t)shots * sizeof(double), hipMemcpyHostToDevice, s.stream));
    {
        KernelScope ks(s, "sample_search", (double)shots * (8.0 + SB * (double)s.amp_bytes()));
        hipLaunchKernelGGL(k_seq_descend<R>, dim3((unsigned)((shots + 255) / 256)), dim3(256), 0, s.stream, psi, B, nblk,
                           w, n, du, shots, dout);
        QFVM_LAUNCHED();
    }
    QFVM_HIP(hipMemcpyAsync(host_out, dout, (size_t)shots * sizeof(uint64_t), hipMemcpyDeviceToHost, s.stream));
    QFVM_HIP(hipStreamSynchronize(s.stream));
}

void sample_sequential_rule(State& s, const double* host_u, int64_t shots, uint64_t* host_out) {
    if (shots <= 0) return;
    uint64_t from = 0;
    double at = 0.0;
    if (s.size >= (uint64_t)SB && (uint64_t)s.size * s.amp_bytes() <= SEQ_BYTES) {
        from = s.dtype == QFVM_C128 ? sample_fast<double>(s, host_u, shots, host_out, &at)
                                    : sample_fast<float>(s, host_u, shots, host_out, &at);
        if (from == NONE) return;
        if (!(at >= SEQ_TINY)) from = 0;  // the loop finds the first nonzero block itself
    }
    if (s.dtype == QFVM_C128)
        sample_typed<double>(s, host_u, shots, host_out, from, at);
    else
        sample_typed<float>(s, host_u, shots, host_out, from, at);
}

}  // namespace qfvm
