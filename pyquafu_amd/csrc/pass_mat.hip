// Fused passes on the matrix cores (complex128, one state).
//
// A pass streams the state through LDS in tiles of 2^b amplitudes (fused.h) and runs its gates in
// groups of three tile qubits. Here a group is not a list of gates but one 8x8 complex matrix per
// value of the few qubits outside the group that its gates depend on (controls, diagonal targets):
// whatever the group's gates are, and however many, a row of 8 amplitudes costs one 8x8 product. As a
// real product that is A X with A = [[Re, -Im], [Im, Re]] interleaved to 16x16 and 16 rows, a column
// block, as X's columns: four v_mfma_f64_16x16x4 per 16 rows.
//
// Operand layout (lane l of the wavefront, kq = l / 16, col = l % 16): X's k step s takes from lane l
// entry 4 s + kq of column col, and the product leaves entry 4 v + kq in register v. The entries of
// A's rows and columns are ordered so that both are component s & 1 of the row's member 2 kq + (s >> 1):
// a lane holds members 2 kq and 2 kq + 1 of row col before and after a product, and gathers and
// scatters them as whole amplitudes.
//
// What bounds it: the matrix cores take 2 cycles per amplitude and group on each of the 1024 SIMDs,
// 0.87 ms per group and 2^30 amplitudes, beside 6.2 ms for the pass's memory traffic, and the two
// overlap only in part. Counters of the 30-qubit, 10-layer benchmark circuit, means over 28 passes of 5 groups
// and 9.1 ms (3.8 TB/s): matrix cores busy 49% of the cycles, vector instructions 20%, LDS 27% (a quarter of
// that bank conflicts), HBM traffic 1.001 times the state's. Its passes take 255 ms, against 317 ms
// in 43 passes on the gate-by-gate kernel; 20 qubits, 20 layers 0.50 against 1.10 ms. The gate-by-gate kernel (k_pass8) spends 0.22 ms per dense gate in vector
// instructions that hide less. complex64 keeps the vector kernels, whose roundings its results are
// compared by.
#include <algorithm>
#include <cstring>

#include "fused.h"

namespace qfvm {

// One gate of a group as the matrix builder applies it. Bits of the 7-bit index: 0..2 the group's
// qubits, 3.. the group's outside qubits.
enum MatKind : int32_t { MK_2X2 = 0, MK_DIAG = 1, MK_SWAP = 2, MK_4X4 = 3 };
struct MatOp {
    int32_t kind;
    int32_t g;    // target bit (MK_DIAG: any bit; MK_4X4: g & 15 is index bit 0, g >> 4 bit 1)
    uint32_t cm;  // control bits, all set
    uint32_t off; // MK_4X4: first entry of the matrix in the pool (complex entries)
    double m[8];
};
struct MatBuild {  // the matrices of one group, one per value of its outside qubits
    int32_t op0, op1;
    int32_t first, count;
};

struct MatGroup {
    int32_t col[4];  // LDS byte offsets (combined by XOR) of the row bits a lane's column stands for,
    int32_t kx[2];   //   of member bits 1 and 2,
    int32_t mx;      //   of member bit 0,
    int32_t cb[2];   //   of the row bits that pick the column block
    int32_t wv[4];   //   and the wavefront
    int32_t voq[4];  // outside qubits beyond the tile: bit j of the matrix index is bit voq[j] of the
                     //   tile's offset (63: none)
    int32_t vcb;     // matrix index bit picked by the column block's upper bit
    int32_t vwv[4];  // and by the wavefront
    uint32_t mat;    // the group's first matrix
};

constexpr int MAT_SEGMENTS = 11;  // runs of qubits outside a tile: at most one more than its high qubits
struct MatPass {
    int b, L, ngroups;
    uint32_t permuted;  // the pass stores its tile with its qubits in other places (FPass::out_bit)
    uint32_t smask[MAT_SEGMENTS];   // tile t sits at the offset sum of (t & smask[i]) << sshift[i]: its
    uint32_t sshift[MAT_SEGMENTS];  //   number's bits on the qubits outside the tile, run by run
    uint32_t lq[10];    // qubit of local bit k (identity below 3)
    uint64_t top[8];    // global offset of amplitude j * threads
    int32_t jx[8];      // and the XOR its number puts on the slot's three lowest bits
    int32_t pslot[10];  // permuted: LDS byte offset of output bit k's source bit,
    int32_t ptop[8];    //   and of output amplitude j * threads' source
    MatGroup g[FUSE_MAX_GROUPS];
};
static_assert(sizeof(MatPass) <= 3072, "kernel argument size");

// LDS layout: amplitude l of the tile in slot l with its three lowest bits XORed by its higher bits
// three at a time. Any three bits that differ modulo 3 then spread eight lanes over all banks, so a
// row order without bank conflicts exists for every group of tiles of 2^12 amplitudes and nearly every
// one of smaller tiles. Linear over XOR.
__host__ __device__ constexpr int mat_slot(int l) { return l ^ (((l >> 3) ^ (l >> 6) ^ (l >> 9) ^ (l >> 12)) & 7); }

typedef double d4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------------------------------------
// Matrix builder: one wavefront per group and eight of its matrices. Lane 8 v + c carries column c of
// the matrix of outside value v through the group's gates in double precision (the gates are the
// same for the whole wavefront, so they are read through the scalar cache), then writes it in the
// order the product's lanes read (64 lanes x 4 steps).
template <int G>
__device__ __forceinline__ void col_2x2(double2 (&v)[8], uint32_t cm, uint32_t hi, const double* __restrict__ m) {
#pragma unroll
    for (int r = 0; r < 8; r++) {
        if ((r >> G) & 1) continue;
        const bool ok = (((uint32_t)r | hi) & cm) == cm;
        const double2 a = v[r], b = v[r | (1 << G)];
        const double2 x = cmul2<double>(mk<double>(m[0], m[1]), a, mk<double>(m[2], m[3]), b);
        const double2 y = cmul2<double>(mk<double>(m[4], m[5]), a, mk<double>(m[6], m[7]), b);
        v[r] = ok ? x : a;
        v[r | (1 << G)] = ok ? y : b;
    }
}

template <int T0, int T1>
__device__ __forceinline__ void col_4x4(double2 (&v)[8], uint32_t cm, uint32_t hi, const double2* __restrict__ m) {
    constexpr int TB = 3 - T0 - T1;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int base = h << TB;
        if ((((uint32_t)base | hi) & cm) != cm) continue;
        double2 x[4], y[4];
#pragma unroll
        for (int k = 0; k < 4; k++) x[k] = v[base | ((k & 1) << T0) | ((k >> 1) << T1)];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            y[r] = cmul<double>(m[4 * r], x[0]);
#pragma unroll
            for (int k = 1; k < 4; k++) {
                const double2 w = m[4 * r + k];
                y[r].x = fma(w.x, x[k].x, fma(-w.y, x[k].y, y[r].x));
                y[r].y = fma(w.x, x[k].y, fma(w.y, x[k].x, y[r].y));
            }
        }
#pragma unroll
        for (int k = 0; k < 4; k++) v[base | ((k & 1) << T0) | ((k >> 1) << T1)] = y[k];
    }
}

__device__ __forceinline__ void col_op(double2 (&v)[8], const MatOp& o, uint32_t hi, const double2* __restrict__ pool) {
    switch (o.kind) {
        case MK_2X2:
            switch (o.g) {
                case 0: col_2x2<0>(v, o.cm, hi, o.m); break;
                case 1: col_2x2<1>(v, o.cm, hi, o.m); break;
                default: col_2x2<2>(v, o.cm, hi, o.m); break;
            }
            break;
        case MK_SWAP: {
#pragma unroll
            for (int g = 0; g < 3; g++) {
                if (o.g != g) continue;
#pragma unroll
                for (int r = 0; r < 8; r++) {
                    if ((r >> g) & 1) continue;
                    const bool ok = (((uint32_t)r | hi) & o.cm) == o.cm;
                    const double2 a = v[r], b = v[r | (1 << g)];
                    v[r] = ok ? b : a;
                    v[r | (1 << g)] = ok ? a : b;
                }
            }
            break;
        }
        case MK_4X4:
            switch (o.g) {
                case 0x10: col_4x4<0, 1>(v, o.cm, hi, pool + o.off); break;
                case 0x01: col_4x4<1, 0>(v, o.cm, hi, pool + o.off); break;
                case 0x20: col_4x4<0, 2>(v, o.cm, hi, pool + o.off); break;
                case 0x02: col_4x4<2, 0>(v, o.cm, hi, pool + o.off); break;
                case 0x21: col_4x4<1, 2>(v, o.cm, hi, pool + o.off); break;
                default: col_4x4<2, 1>(v, o.cm, hi, pool + o.off); break;
            }
            break;
        default:  // MK_DIAG
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const uint32_t i = (uint32_t)r | hi;
                if ((i & o.cm) != o.cm) continue;
                const bool one = (i >> o.g) & 1u;
                v[r] = cmul<double>(one ? mk<double>(o.m[6], o.m[7]) : mk<double>(o.m[0], o.m[1]), v[r]);
            }
    }
}

__global__ void __launch_bounds__(64) k_mat_build(const MatBuild* __restrict__ todo, const MatOp* __restrict__ ops,
                                                  const double2* __restrict__ pool, double* __restrict__ out) {
    const MatBuild t = todo[blockIdx.x];
    const int var = (int)blockIdx.y * 8 + (int)(threadIdx.x >> 3), c = threadIdx.x & 7;
    if ((int)blockIdx.y * 8 >= t.count) return;
    double2 v[8];
#pragma unroll
    for (int r = 0; r < 8; r++) v[r] = mk<double>(r == c ? 1.0 : 0.0, 0.0);
    const uint32_t hi = (uint32_t)var << 3;
    MatOp next = ops[t.op0];  // the array ends with a spare record
    for (int k = t.op0; k < t.op1; k++) {
        const MatOp o = next;
        next = ops[k + 1];
        col_op(v, o, hi, pool);
    }
    if (var >= t.count) return;
    const int mi = t.first + var;
    double* dst = out + (size_t)mi * 256;
    const int kq = c >> 1, s = (c & 1) << 1;
#pragma unroll
    for (int r = 0; r < 8; r++)
#pragma unroll
        for (int rc = 0; rc < 2; rc++) {
            const int i = 4 * (((r & 1) << 1) | rc) + (r >> 1);  // output component rc of member r
            double* at = dst + (size_t)(i + 16 * kq) * 4 + s;    // columns: both components of member c
            at[0] = rc ? v[r].y : v[r].x;
            at[1] = rc ? v[r].x : -v[r].y;
        }
}

// ------------------------------------------------------------------------------------------------
// orders LDS traffic between the wavefronts of a workgroup; loads into registers stay in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// HBM -> LDS loads of a thread's eight amplitudes: slot j NT + tid takes amplitude
// mat_slot(j NT + tid) = (j NT + mat_slot(tid)) ^ jx[j], whose offset starts from g = that of
// mat_slot(tid). AUX is the instruction's cache policy (2: non-temporal)
template <int AUX>
__device__ __forceinline__ void load_tile(const double2* __restrict__ psi, unsigned char* lds, const MatPass& pd,
                                          uint64_t g, int NT, int wave) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const void* src = (const void*)(psi + ((g ^ (uint64_t)pd.jx[j]) | pd.top[j]));
        auto* dst = (__attribute__((address_space(3))) void*)(lds + (size_t)(j * NT + wave * 64) * 16);
        __builtin_amdgcn_global_load_lds(src, dst, 16, 0, AUX);
    }
}

// global offset of a tile
__device__ __forceinline__ uint64_t mat_base(uint32_t tile, const MatPass& pd) {
    uint64_t base = 0;
#pragma unroll
    for (int k = 0; k < MAT_SEGMENTS; k++) base |= (uint64_t)(tile & pd.smask[k]) << pd.sshift[k];
    return base;
}
// and of a local index below the thread count, within the tile
__device__ __forceinline__ uint64_t mat_local(int l, const MatPass& pd) {
    uint64_t g = (uint64_t)(l & 7);
#pragma unroll
    for (int k = 3; k < 10; k++) g |= (uint64_t)((l >> k) & 1) << pd.lq[k];
    return g;
}

// One group as a lane sees it: the LDS offset of its member 0 in column block 0, the uniform offsets
// of the other member and blocks, and the wavefront's matrix (of column blocks 0 and 1).
struct MatCursor {
    int sl, mx, cb0, cb1, vcb;
    const double* mat;
    d4 a;
};
__device__ __forceinline__ MatCursor mat_open(const MatGroup& G, uint64_t base, int wave, int lane,
                                              const double* __restrict__ mats) {
    MatCursor c;
    auto bit = [&](int k) { return -((lane >> k) & 1); };
    c.sl = (bit(0) & G.col[0]) ^ (bit(1) & G.col[1]) ^ (bit(2) & G.col[2]) ^ (bit(3) & G.col[3]) ^ (bit(4) & G.kx[0]) ^
           (bit(5) & G.kx[1]);
    int sw = 0, v = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        sw ^= ((wave >> j) & 1) ? G.wv[j] : 0;
        v |= (((wave >> j) & 1) ? G.vwv[j] : 0) | ((int)((base >> G.voq[j]) & 1) << j);
    }
    c.sl ^= sw;
    c.mx = G.mx;
    c.cb0 = G.cb[0];
    c.cb1 = G.cb[1];
    c.vcb = G.vcb * 256;
    c.mat = mats + (size_t)(G.mat + (uint32_t)v) * 256 + lane * 4;
    c.a = *reinterpret_cast<const d4*>(c.mat);
    return c;
}

// A wavefront's four column blocks of a group: their LDS offsets and this lane's members.
struct MatRows {
    double2 x[4][2];
    int at[4];
};
__device__ __forceinline__ void mat_gather(const unsigned char* lds, const MatCursor& c, MatRows& w) {
#pragma unroll
    for (int cb = 0; cb < 4; cb++) {
        w.at[cb] = c.sl ^ ((cb & 1) ? c.cb0 : 0) ^ ((cb & 2) ? c.cb1 : 0);
        w.x[cb][0] = *reinterpret_cast<const double2*>(lds + w.at[cb]);
        w.x[cb][1] = *reinterpret_cast<const double2*>(lds + (w.at[cb] ^ c.mx));
    }
}
// Multiplies column blocks cb and cb + 1 by a and stores them (every row belongs to one wavefront and one
// block, so nothing else reads them before the barrier); whether a lane's first products are finite.
// The first and the last two k steps are summed apart and added: the partial sums are half as long, and
// with them the product's rounding (error of the state after 40 layers on 16 qubits 2.12e-15 with
// one sum, 1.95e-15 with two, 1.90e-15 with four; 1.89e-15 on the vector kernels). Two blocks at a time two
// sums cost nothing (30 qubits, 10 layers: 260.0 ms with one, 254.9 with two; four take 4% more).
__device__ __forceinline__ bool mat_pair(unsigned char* lds, const MatRows& w, int mx, int cb, const d4& a) {
    d4 sum[2][2];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const double b = s ? w.x[cb + k][h].y : w.x[cb + k][h].x;
                sum[k][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[2 * h + s], b, s ? sum[k][h] : d4{0, 0, 0, 0}, 0, 0, 0);
            }
    bool fin = true;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const d4 r = sum[k][0] + sum[k][1];
        *reinterpret_cast<double2*>(lds + w.at[cb + k]) = make_double2(r[0], r[1]);
        *reinterpret_cast<double2*>(lds + (w.at[cb + k] ^ mx)) = make_double2(r[2], r[3]);
        fin = fin & __builtin_isfinite(r[0]);
    }
    return fin;
}

// The same products entry by entry, skipping the matrix's zeros (see k_pass_mat), stored.
__device__ __forceinline__ void mat_sparse(unsigned char* lds, const MatCursor& c, const MatGroup& G, int lane) {
    const int kq = lane >> 4, kx0 = G.kx[0], kx1 = G.kx[1];
#pragma unroll 1
    for (int cb = 0; cb < 4; cb++) {
        const int at = c.sl ^ ((cb & 1) ? c.cb0 : 0) ^ ((cb & 2) ? c.cb1 : 0);
        const int row = at ^ ((kq & 1) ? kx0 : 0) ^ ((kq & 2) ? kx1 : 0);  // slot of member 0
        const double* a = c.mat - lane * 4 + ((cb & 2) ? c.vcb : 0);
        double2 y[2] = {{0.0, 0.0}, {0.0, 0.0}};
#pragma unroll 1
        for (int m = 0; m < 8; m++) {
            const double2 x = *reinterpret_cast<const double2*>(
                lds + (row ^ ((m & 1) ? c.mx : 0) ^ ((m & 2) ? kx0 : 0) ^ ((m & 4) ? kx1 : 0)));
#pragma unroll
            for (int r = 0; r < 2; r++) {  // member 2 kq + r of the result
                const double* w = a + (8 * r + kq + 16 * (m >> 1)) * 4 + ((m & 1) << 1);
                const double re = w[0], im = -w[1];
                if (re != 0.0) {
                    y[r].x = fma(re, x.x, y[r].x);
                    y[r].y = fma(re, x.y, y[r].y);
                }
                if (im != 0.0) {
                    y[r].x = fma(-im, x.y, y[r].x);
                    y[r].y = fma(im, x.x, y[r].y);
                }
            }
        }
        // (the wavefront has read the block's rows; no other block holds them)
        *reinterpret_cast<double2*>(lds + at) = y[0];
        *reinterpret_cast<double2*>(lds + (at ^ c.mx)) = y[1];
    }
}

__device__ __forceinline__ void mat_put(double2* p, double2 v, int nt) {
    typedef double d2 __attribute__((ext_vector_type(2)));
    const d2 w = {v.x, v.y};
    if (nt)
        __builtin_nontemporal_store(w, reinterpret_cast<d2*>(p));
    else
        *reinterpret_cast<d2*>(p) = w;
}

// Stores the tile; a permuted one amplitude e from its source's slot.
__device__ __forceinline__ void store_tile(double2* __restrict__ psi, const unsigned char* lds, const MatPass& pd,
                                           uint64_t g, int tid, int NT, int nt) {
    __builtin_amdgcn_s_setprio(2);
    if (pd.permuted) {
        int st = 0;
#pragma unroll
        for (int k = 0; k < 10; k++) st ^= -((tid >> k) & 1) & pd.pslot[k];
#pragma unroll
        for (int j = 0; j < 8; j++)
            mat_put(&psi[g | pd.top[j]], *reinterpret_cast<const double2*>(lds + (st ^ pd.ptop[j])), nt);
    } else {
        const int su = mat_slot(tid);
#pragma unroll
        for (int j = 0; j < 8; j++)
            mat_put(&psi[g | pd.top[j]], *reinterpret_cast<const double2*>(lds + (size_t)((j * NT + su) ^ pd.jx[j]) * 16), nt);
    }
    __builtin_amdgcn_s_setprio(0);
}

// One tile per workgroup of 2^(b-3) threads; wavefront w holds rows 64 w .. 64 w + 63 of every group
// (in the group's own row order) as four column blocks. `nt`: the state is far larger than the
// caches, so its lines are loaded and stored with the non-temporal hint.
// The matrix cores multiply every entry, so an infinity or a NaN reaches all members of its row (0 * inf),
// though gates as X, CX, CZ and diagonal ones only move or scale amplitudes. Such a row has no finite
// product from then on; so the last group's products tell, and before anything is stored the tile is loaded
// again and multiplied without the matrices' zeros (a flag after the tile; correcting each group's products
// on the spot took 5% of the 30-qubit circuit).
// LARGE (states of 2^24 amplitudes and more): wavefronts whose blocks take one matrix and those with two have
// code of their own, and only the last group tests its products: 28 qubits, 6 layers 32.2 -> 31.2 ms, 26
// qubits 7.08 -> 6.84. Smaller states wait for each tile's chain of groups instead, and the shorter code is
// the faster one there (16 qubits, 3 layers 75.1 us against 77.2).
template <bool LARGE>
__global__ void __launch_bounds__(1024) k_pass_mat(double2* __restrict__ psi, const MatPass pd,
                                                   const double* __restrict__ mats, int nt) {
    extern __shared__ unsigned char lds[];
    const int tid = threadIdx.x, NT = blockDim.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint64_t base = mat_base(blockIdx.x, pd);
    const uint64_t g_sw = base | mat_local(mat_slot(tid), pd);
    int* again = reinterpret_cast<int*>(lds + (size_t)NT * 128);
    __builtin_amdgcn_s_setprio(2);
    if (nt)
        load_tile<2>(psi, lds, pd, g_sw, NT, wave);
    else
        load_tile<0>(psi, lds, pd, g_sw, NT, wave);
    __builtin_amdgcn_s_setprio(0);
    if (tid == 0) *again = 0;
    MatCursor cur{};
    if (pd.ngroups > 0) cur = mat_open(pd.g[0], base, wave, lane, mats);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (int gi = 0; gi < pd.ngroups; gi++) {
        MatRows w;
        mat_gather(lds, cur, w);
        const int mx = cur.mx;
        bool finite;
        const MatGroup& next = pd.g[gi + 1 < pd.ngroups ? gi + 1 : gi];  // its matrix arrives over the barrier
        if (LARGE && cur.vcb == 0) {  // one matrix for the wavefront
            const d4 a = cur.a;
            finite = mat_pair(lds, w, mx, 0, a);
            cur = mat_open(next, base, wave, lane, mats);
            finite = mat_pair(lds, w, mx, 2, a) & finite;
        } else {
            d4 a = cur.a;
            if (LARGE || cur.vcb) a = *reinterpret_cast<const d4*>(cur.mat + cur.vcb);
            finite = mat_pair(lds, w, mx, 0, cur.a);
            cur = mat_open(next, base, wave, lane, mats);
            finite = mat_pair(lds, w, mx, 2, a) & finite;
        }
        if ((!LARGE || gi + 1 == pd.ngroups) && !__all(finite) && lane == 0) *again = 1;
        lds_barrier();
    }
    int t = tid;
    asm volatile("" : "+v"(t));  // (offsets are formed anew: kept over the groups, they would not fit the registers)
    if (__builtin_amdgcn_readfirstlane(*again)) {
        __syncthreads();
        load_tile<0>(psi, lds, pd, base | mat_local(mat_slot(t), pd), NT, wave);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
#pragma unroll 1
        for (int gi = 0; gi < pd.ngroups; gi++) {
            mat_sparse(lds, mat_open(pd.g[gi], base, wave, lane, mats), pd.g[gi], lane);
            __syncthreads();
        }
    }
    store_tile(psi, lds, pd, base | mat_local(t, pd), t, NT, nt);
}

// ------------------------------------------------------------------------------------------------
// LDS byte offset of tile-local bit k
static int slot_of_bit(int k) { return mat_slot(1 << k) * 16; }

namespace {
struct MatPlanData {
    std::vector<MatOp> ops;
    std::vector<cd> pool;
    std::vector<MatBuild> todo;
    uint32_t matrices = 0;
};
}  // namespace

// The pass's kernel argument; its groups' gates go to d.ops and its matrices to d.todo.
static MatPass encode_mat_pass(const State& s, const FPass& p, MatPlanData& d) {
    const int b = (int)p.Q.size();
    int L = 0;
    while (L < b && p.Q[(size_t)L] == L) L++;
    MatPass pd{};
    if ((int)p.groups.size() > FUSE_MAX_GROUPS || b < 9 || b > 13 || b > s.n || L < 3 || p.group_bits != 3)
        throw Error(QFVM_ERR_RUNTIME, "matrix-core pass exceeds kernel limits");
    pd.b = b;
    pd.L = L;
    pd.ngroups = (int)p.groups.size();
    int local_of[64];
    for (int k = 0; k < 64; k++) local_of[k] = -1;
    for (int k = 0; k < b; k++) local_of[p.Q[(size_t)k]] = k;
    for (int k = 0; k < 10 && k < b; k++) pd.lq[k] = (uint32_t)p.Q[(size_t)k];
    for (int q = 0, k = 0, run = -1; q < s.n; q++) {  // k: bit of the tile number
        if (local_of[q] >= 0) {
            if (k > 0 && q > 0 && local_of[q - 1] < 0) run++;
            continue;
        }
        if (run < 0) run = 0;
        if (run >= MAT_SEGMENTS) throw Error(QFVM_ERR_RUNTIME, "tile with too many runs of qubits");
        pd.smask[run] |= 1u << k;
        pd.sshift[run] = (uint32_t)(q - k);
        k++;
    }
    for (int j = 0; j < 8; j++) {
        for (int i = 0; i < 3; i++)
            if ((j >> i) & 1) pd.top[j] |= 1ull << p.Q[(size_t)(b - 3 + i)];
        const int l = j << (b - 3);
        pd.jx[j] = mat_slot(l) ^ l;
    }
    const int waves_bits = b - 9;
    for (int gi = 0; gi < pd.ngroups; gi++) {
        const FGroup& G = p.groups[(size_t)gi];
        MatGroup& mg = pd.g[gi];
        uint64_t S = 0, ext = 0;
        for (int j = 0; j < 3; j++) {
            if (G.stage || G.S[j] < 0 || local_of[G.S[j]] < 0) throw Error(QFVM_ERR_RUNTIME, "group qubit outside the tile");
            S |= 1ull << G.S[j];
        }
        for (const FOpHost& o : G.ops) {
            ext |= o.cm_ext;
            if (o.kind == F_PHASE) ext |= 1ull << o.g;
        }
        if ((ext & S) || __builtin_popcountll(ext) > MAT_MAX_EXT) throw Error(QFVM_ERR_RUNTIME, "group with too many outside qubits");
        // member bits: bit j <-> G.S[j]
        int member[3];
        for (int j = 0; j < 3; j++) member[j] = local_of[G.S[j]];
        mg.mx = slot_of_bit(member[0]);
        mg.kx[0] = slot_of_bit(member[1]);
        mg.kx[1] = slot_of_bit(member[2]);
        // variant bits in ascending qubit order
        int vbit[64];
        int nv = 0;
        std::vector<int> in_tile, rows;  // local bits of the rows: outside qubits of the group, others
        for (int j = 0; j < 4; j++) mg.voq[j] = 63;
        for (int q = 0; q < s.n; q++) {
            vbit[q] = -1;
            if ((ext >> q) & 1) {
                vbit[q] = nv;
                if (local_of[q] >= 0)
                    in_tile.push_back(local_of[q]);
                else
                    mg.voq[nv] = q;
                nv++;
            } else if (local_of[q] >= 0 && !((S >> q) & 1)) {
                rows.push_back(local_of[q]);
            }
        }
        if (rows.size() < 5) throw Error(QFVM_ERR_RUNTIME, "group with too many outside qubits in the tile");
        // column bits: a lane's four; one of each class modulo 3 first (no bank conflicts)
        std::vector<int> cols;
        auto take = [&](auto&& want) {
            for (size_t i = 0; i < rows.size(); i++)
                if (want(rows[i])) {
                    cols.push_back(rows[i]);
                    rows.erase(rows.begin() + (std::ptrdiff_t)i);
                    return;
                }
        };
        for (int cls = 0; cls < 3; cls++) take([&](int k) { return k % 3 == cls; });
        while (cols.size() < 4) take([](int) { return true; });
        for (int j = 0; j < 4; j++) mg.col[j] = slot_of_bit(cols[(size_t)j]);
        // the other rows: column blocks take plain row bits while there are any (one matrix for the
        // wavefront), wavefronts the group's outside qubits
        std::vector<int> rest = rows;
        rest.insert(rest.end(), in_tile.begin(), in_tile.end());
        if ((int)rest.size() != 2 + waves_bits) throw Error(QFVM_ERR_RUNTIME, "row bits of a matrix-core group");
        auto variant_of = [&](int local) {
            const int v = vbit[p.Q[(size_t)local]];
            return v >= 0 ? 1 << v : 0;
        };
        for (int j = 0; j < 2; j++) mg.cb[j] = slot_of_bit(rest[(size_t)j]);
        mg.vcb = variant_of(rest[1]);
        for (int j = 0; j < waves_bits; j++) {
            mg.wv[j] = slot_of_bit(rest[(size_t)(2 + j)]);
            mg.vwv[j] = variant_of(rest[(size_t)(2 + j)]);
        }
        auto index_bits = [&](uint64_t qubits) {
            uint32_t m = 0;
            for (uint64_t x = qubits; x; x &= x - 1) m |= 8u << vbit[__builtin_ctzll(x)];
            return m;
        };
        const int op0 = (int)d.ops.size();
        for (const FOpHost& o : G.ops) {
            MatOp r{};
            r.cm = o.cm_group | index_bits(o.cm_ext);
            r.g = o.kind == F_PHASE ? 3 + vbit[o.g] : o.g;
            for (int k = 0; k < 4; k++) {
                r.m[2 * k] = o.m[k].real();
                r.m[2 * k + 1] = o.m[k].imag();
            }
            switch (o.kind) {
                case F_DENSE:
                case F_REAL: r.kind = MK_2X2; break;
                case F_DIAG:
                case F_PHASE: r.kind = MK_DIAG; break;
                case F_SWAP: r.kind = MK_SWAP; break;
                case F_DENSE4:
                    if (o.mx.size() != 16 || o.g == o.target) throw Error(QFVM_ERR_RUNTIME, "malformed 4x4 op");
                    r.kind = MK_4X4;
                    r.g = o.g | (o.target << 4);
                    r.off = (uint32_t)d.pool.size();
                    d.pool.insert(d.pool.end(), o.mx.begin(), o.mx.end());
                    break;
                default: throw Error(QFVM_ERR_RUNTIME, "op kind not supported by matrix-core passes");
            }
            d.ops.push_back(r);
        }
        mg.mat = d.matrices;
        d.todo.push_back(MatBuild{op0, (int)d.ops.size(), (int)d.matrices, 1 << nv});
        d.matrices += 1u << nv;
    }
    if (!p.out_bit.empty()) {
        if ((int)p.out_bit.size() != b) throw Error(QFVM_ERR_RUNTIME, "qubit permutation outside its pass");
        pd.permuted = 1;
        int from[FUSE_MAX_TILE_BITS];
        for (int k = 0; k < b; k++) from[k] = -1;
        for (int k = 0; k < b; k++) {
            const int o = p.out_bit[(size_t)k];
            if (o < 0 || o >= b || from[o] >= 0) throw Error(QFVM_ERR_RUNTIME, "tile qubit permutation is not a permutation");
            from[o] = k;
        }
        for (int k = 0; k < b - 3; k++) pd.pslot[k] = slot_of_bit(from[k]);
        for (int j = 0; j < 8; j++)
            for (int i = 0; i < 3; i++)
                if ((j >> i) & 1) pd.ptop[j] ^= slot_of_bit(from[b - 3 + i]);
    }
    return pd;
}

// matrices built at a time (bounds the buffer: 64 MiB at complex128)
constexpr uint32_t MAT_LIMIT = 1u << 15;

void execute_mat_plan(State& s, const std::vector<PlanItem>& plan) {
    if (s.dtype != QFVM_C128) throw Error(QFVM_ERR_RUNTIME, "matrix-core passes are complex128");
    size_t i = 0;
    while (i < plan.size()) {
        // a segment of the plan: its gates are uploaded and its matrices built in one launch
        MatPlanData d;
        std::vector<MatPass> passes;
        size_t e = i;
        for (; e < plan.size() && d.matrices < MAT_LIMIT; e++)
            if (plan[e].fused) passes.push_back(encode_mat_pass(s, plan[e].pass, d));
        double* mats = nullptr;
        if (!d.todo.empty()) {
            d.ops.push_back(MatOp{});  // the builder reads one record ahead
            const size_t obytes = d.ops.size() * sizeof(MatOp);
            const size_t toff = (obytes + 255) / 256 * 256;
            const size_t poff = (toff + d.todo.size() * sizeof(MatBuild) + 255) / 256 * 256;
            const size_t bytes = poff + d.pool.size() * sizeof(cd);
            unsigned char* host = s.stage_host(STAGE_PLAN, bytes);
            unsigned char* dev = s.stage_dev(STAGE_PLAN, bytes);
            mats = reinterpret_cast<double*>(s.ensure_ops((size_t)d.matrices * 256 * sizeof(double)));
            std::memcpy(host, d.ops.data(), obytes);
            std::memcpy(host + toff, d.todo.data(), d.todo.size() * sizeof(MatBuild));
            if (!d.pool.empty()) std::memcpy(host + poff, d.pool.data(), d.pool.size() * sizeof(cd));
            s.stage_upload(STAGE_PLAN, bytes);
            KernelScope ks(s, "mat_build", (double)bytes + (double)d.matrices * 256 * sizeof(double));
            hipLaunchKernelGGL(k_mat_build, dim3((unsigned)d.todo.size(), (1u << MAT_MAX_EXT) / 8), dim3(64), 0,
                               s.stream, reinterpret_cast<const MatBuild*>(dev + toff),
                               reinterpret_cast<const MatOp*>(dev), reinterpret_cast<const double2*>(dev + poff), mats);
            QFVM_LAUNCHED();
        }
        size_t k = 0;
        for (; i < e; i++) {
            if (!plan[i].fused) {
                launch_gate(s, plan[i].gate);
                continue;
            }
            const MatPass& pd = passes[k++];
            const size_t lds = ((size_t)1 << pd.b) * sizeof(double2) + sizeof(double2);  // and k_pass_mat's flag
            const unsigned threads = (1u << pd.b) >> 3;
            const auto fn = s.n >= 24 ? k_pass_mat<true> : k_pass_mat<false>;
            if (lds > 65536) allow_large_lds(reinterpret_cast<const void*>(fn), s.device);
            const int nt = s.size * sizeof(double2) > (256ull << 20) ? 1 : 0;
            KernelScope ks(s, "fused_pass", 2.0 * (double)s.size * sizeof(double2));
            hipLaunchKernelGGL(fn, dim3((unsigned)(1ull << (s.n - pd.b))), dim3(threads), lds, s.stream,
                               reinterpret_cast<double2*>(s.psi), pd, mats, nt);
            QFVM_LAUNCHED();
        }
    }
}

}  // namespace qfvm
