// steppe_amd/csrc/f2_split.hip — per-block f2 from fixed-point 8-bit digits on int8 MFMA.
//
// The reference's default precision is cuBLAS's closed FP64 emulation on integer
// units (src/device/cuda/f2_block_kernel.cu:121-144).  This is an independent
// construction from the published Ozaki-scheme idea (Ozaki, Ogita, Oishi & Rump,
// Numer. Algorithms 59:95-118, 2012; Ootomo, Ozaki & Yokota, IJHPCA 2024): split
// every operand into fixed-point digits whose pairwise products and partial sums
// are exact in the MFMA's int32 accumulator, and recombine the exact partial sums
// in FP64.  It computes the same estimator as the FP64 path (f2_fp64.hip):
//
//   num_ij = sum_s v_i v_j [(q_i - q_j)^2 - h_i - h_j],  f2 = num / vpair
//
// Operands.  The estimator only sees differences q_i - q_j, so any per-SNP shift of q
// leaves it unchanged; with q' = q - 1/2 (|q'| <= 1/2) and w = -(q'^2 - h)/2
// (|w| <= 1/8), both as 48-bit integers in six balanced 8-bit digits:
//   q~ = 2^-7 sum_k d_k 2^-8k,           |q~ - q'| <= 2^-48;
//   w~ = -128 sum_k W_k 2^(-14-8k)       (computed from q~), |w~ - w| <= 2^-48.
// With level units U_t = 2^(-14-8t) and V = -128 v,
//   -num_ij / 2 = sum_s [ q~_i q~_j + w~_i v_j + v_i w~_j ] = sum_t U_t * L_t,
//   L_t = sum_s [ sum_{k+l=t} d_k(i) d_l(j) + W_t(i) V(j) + V(i) W_t(j) ],  t = 0..5.
// Products with k + l >= 6 are dropped (<= 2^-45 per SNP).
//
// V has no plane of its own: |W_0| <= 16, so W_0 + 96 is stored for an observed entry (a
// byte in [79, 113]: bit 6 is set) and 0 for a missing one, and V = -128 v is the byte
// (W_0' << 1) & 0x80.  The offset adds 96 (v_i V_j + V_i v_j) = -24576 v_i v_j per SNP
// to L_0, which the epilogue takes back from the pair count, in integers.
//
// Per SNP, |L_5| grows by at most 2*64*128 + 4*2^14 + 2*2^14 = 114,688 and the others by
// less, so 16,384 SNPs keep every level below 2^31: a block accumulates in six int32
// words per output with no carries, and FP64 appears only in the epilogue.  Longer blocks
// are summed in segments of 16,384 SNPs, whose FP64 partial sums meet in the f2 tensor.
//
// MFMA work per (pair, SNP): 33 int8 products (21 digit by digit, 12 digit by V) at twice
// the BF16 rate, plus the pair count V V^T in a kernel of its own.  Operand bytes per
// (population, SNP): 12.  (The same scheme on BF16 / FP16 digits with FP32 accumulators
// took 29 products at the BF16 rate, 22 bytes, and carries every 128 SNPs.)
//
// Kernel shape: persistent workgroups of 8 wavefronts (2 per SIMD) own a 128x128
// output tile of one jackknife block; each wavefront owns 64x32 (two 32x32 MFMA
// tiles, six int32 accumulators per output).  Each 32-SNP K-step is two phases (the q
// digits, then the w digits) whose 48 KB of planes arrive in a ring of three LDS slots
// by direct global->LDS loads, issued two phases ahead.
//
// Bound and measured: the contraction issues 33 x 2 ops per output and SNP of its sub-tiles
// (blocks padded to 64 SNPs; of a diagonal tile ten of sixteen sub-tiles), 1.10 times those of
// the population pairs.  1000 populations x 1.2M SNPs: 4.36e13 ops in 18.6 ms = 2.34 POP/s
// with the matrix pipes busy 64% of the cycles, 94% of the rate that a plain 8192^3 int8
// library product reaches on this card (2.49); 1000 x 597,573: 9.2 ms, on the BF16 / FP16
// digits 18.3.  Prep writes 12 instead of 23 bytes per entry: 2.0 instead of 4.5 ms.

#include <utility>

#include "common.hpp"
#include "f2_layout.hpp"

namespace stp {

void launch_zero_u32(unsigned* p, int n, hipStream_t st);

namespace {

typedef int i4 __attribute__((ext_vector_type(4)));
typedef int i16v __attribute__((ext_vector_type(16)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));

constexpr int kPlanes = kSplitPlanes;  // d0..d5 (0-5), W0'..W5 (6-11)
constexpr int kSetPlanes = 6;          // planes of one phase: the q digits or the w digits
constexpr int kChunk = 1024;           // bytes per (32-row group, 32-SNP step, plane)
constexpr int kGroups = 8;             // 32-row groups per workgroup tile: 4 left + 4 right
constexpr int kSlotBytes = kGroups * kSetPlanes * kChunk;   // 48 KB
constexpr int kWaves = 8;
constexpr int kW0Offset = 96;                               // W_0' - W_0 of an observed entry
constexpr int kL0PerPair = 2 * 128 * kW0Offset;             // what it takes from L_0 per pair and SNP
constexpr int kSegSteps = 512;                              // K-steps whose level sums fit int32

// f(std::integral_constant<int, I>) for I = 0 .. N-1, as straight-line code.
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (f(std::integral_constant<int, I>{}), ...);
    }(std::make_integer_sequence<int, N>{});
}

// ---------------------------------------------------------------------------------
// prep: frequencies -> 12 digit planes in 32x32x32 MFMA fragment order, in one pass:
//   plane chunk (g32, t32, p) holds rows 32 g32 + lane%32, SNPs 32 t32 + 16 (lane/32) + j
//   at byte offset ((g32 * KS32 + t32) * 12 + p) * 1024 + lane * 16 + j.
// A workgroup converts one (32-row group, 64-SNP chunk) unit at a time: it stages each
// entry's two 48-bit integers in LDS (12 bytes, from coalesced row reads), then every
// thread transposes the bytes of one 16-SNP fragment of the q or the w digits into six
// 16-byte stores.
// ---------------------------------------------------------------------------------
constexpr int kStageLd = 65;  // LDS row stride (dwords) of the staged unit

// The staged unit: per entry bytes 0-3 of the q integer, its bytes 4-5 with the w
// integer's bytes 4-5 above them, bytes 0-3 of the w integer.
struct Stage {
    unsigned q[32 * kStageLd];
    unsigned t[32 * kStageLd];
    unsigned w[32 * kStageLd];
};

// An integer |x| < 2^47 given as a double (rounded to nearest even): its balanced digits
// in bytes 0 (least significant) to 4, each in [-128, 127], and the rest in byte 5.
// Adding 1.5 * 2^52 leaves the integer in the low bits; adding 128 to every lower digit
// place makes plain bytes of the balanced digits, and flipping each top bit undoes it.
__device__ inline unsigned long long balanced48(double x) {
    const unsigned long long bits = static_cast<unsigned long long>(__double_as_longlong(x + 0x1.8p52));
    return (bits + 0x8080808080ull) ^ 0x8080808080ull;
}

// Stage one entry; h < 0 or NaN (a frequency outside [0, 1]) counts as missing.
__device__ inline void stage_entry(Stage& st, int at, bool ok, double q, double nm1) {
    unsigned long long Q = 0, W = 0;
    const double h = q * (1.0 - q) / (nm1 > 1.0 ? nm1 : 1.0);
    if (ok && h >= 0.0) {
        const double x = (q - 0.5) * 0x1p47;
        const double qt = ((x + 0x1.8p52) - 0x1.8p52) * 0x1p-47;
        Q = balanced48(x);
        W = balanced48((qt * qt - h) * 0x1p46) + (static_cast<unsigned long long>(kW0Offset) << 40);
    }
    st.q[at] = static_cast<unsigned>(Q);
    st.t[at] = (static_cast<unsigned>(Q >> 32) & 0xFFFFu) | (static_cast<unsigned>(W >> 32) << 16);
    st.w[at] = static_cast<unsigned>(W);
}

// Staging reads of the two frequency sources.  Each thread stages 8 elements of the
// 32 x 64 unit: fetch() issues the global loads into registers (so a workgroup can
// fetch its next unit while it converts the current one), put() turns them into staged
// entries with h = q(1-q)/max(n-1, 1) as in the reference's het_correction
// (src/core/internal/f2_estimator.hpp:22-29).
struct CountsSrc {
    const std::uint16_t* a2;
    const std::uint16_t* n;
    std::int64_t ld;
    struct Raw {
        unsigned a[8], c[8];
        bool ok[8];
    };
    // Lanes run along the SNP axis: each wavefront reads 128 contiguous bytes per row.
    // The loads are unconditional (entries outside the unit re-read a valid one and are
    // masked), so the compiler knows how many are in flight and waits for them alone,
    // not for the previous unit's plane stores as well.
    __device__ Raw fetch(int r0, int P, std::int64_t snp0, int live, int tid) const {
        Raw raw;
        const int kk = tid & 63;
        const bool col_ok = kk < live;
        const std::int64_t col = snp0 + (col_ok ? kk : 0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = (tid >> 6) + 4 * i;
            const bool ok = col_ok && r0 + row < P;
            const std::int64_t o = static_cast<std::int64_t>(ok ? r0 + row : r0) * ld + col;
            raw.a[i] = a2[o];
            raw.c[i] = n[o];
            raw.ok[i] = ok;
        }
        return raw;
    }
    __device__ void put(const Raw& raw, int tid, Stage& st) const {
        const int kk = tid & 63;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = (tid >> 6) + 4 * i;
            const double nd = static_cast<double>(raw.c[i]);
            const bool ok = raw.ok[i] && raw.c[i];
            const double q = static_cast<double>(raw.a[i]) / (ok ? 2.0 * nd : 1.0);
            stage_entry(st, row * kStageLd + kk, ok, q, nd - 1.0);
        }
    }
};

struct QvnSrc {
    const double* q;
    const double* v;
    const double* n;
    struct Raw {
        double q[8], v[8], n[8];
        bool ok[8];
    };
    // Q/V/N are population-fastest (i + P*s): lanes run along the population axis.
    // Unconditional loads, as in CountsSrc::fetch.
    __device__ Raw fetch(int r0, int P, std::int64_t snp0, int live, int tid) const {
        Raw raw;
        const int row = tid & 31;
        const bool row_ok = r0 + row < P;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int kk = (tid >> 5) + 8 * i;
            const bool ok = row_ok && kk < live;
            const std::int64_t o = (row_ok ? r0 + row : r0) + static_cast<std::int64_t>(P) * (snp0 + (ok ? kk : 0));
            raw.v[i] = v[o];
            raw.q[i] = q[o];
            raw.n[i] = n[o];
            raw.ok[i] = ok;
        }
        return raw;
    }
    __device__ void put(const Raw& raw, int tid, Stage& st) const {
        const int row = tid & 31;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            stage_entry(st, row * kStageLd + (tid >> 5) + 8 * i, raw.ok[i] && raw.v[i] != 0.0, raw.q[i],
                        raw.n[i] - 1.0);
    }
};

// Rows, SNP range and block of a prep unit (32-row group, 64-SNP chunk).
struct PrepUnit {
    int g, live;
    std::int64_t c, snp0;
};

// The block-table arrays arrive as separate read-only, non-aliased kernel arguments, so
// that these uniform lookups compile to scalar loads: a vector load here would have to
// wait (in order) for the previous unit's plane stores before its value could be used.
__device__ inline PrepUnit prep_unit(std::int64_t u, std::int64_t n_chunks, const std::int64_t* __restrict__ s0,
                                     const std::int32_t* __restrict__ len, const std::int64_t* __restrict__ k0,
                                     const std::int32_t* __restrict__ chunk_block) {
    PrepUnit pu;
    pu.g = static_cast<int>(u / n_chunks);
    pu.c = u - static_cast<std::int64_t>(pu.g) * n_chunks;
    const int b = chunk_block[pu.c];
    const std::int64_t local0 = 64 * pu.c - k0[b];
    pu.snp0 = s0[b] + local0;
    pu.live = static_cast<int>(max<std::int64_t>(0, min<std::int64_t>(64, len[b] - local0)));
    return pu;
}

// Workgroup barrier for the LDS stage only: waits for this wavefront's LDS operations,
// not for its outstanding global stores (__syncthreads would also wait for those).
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Byte columns of four dwords: out[i] = byte i of x[0], x[1], x[2], x[3].
__device__ inline void bytes4x4(const unsigned (&x)[4], unsigned (&out)[4]) {
    const unsigned a01 = __builtin_amdgcn_perm(x[1], x[0], 0x05010400u);
    const unsigned b01 = __builtin_amdgcn_perm(x[1], x[0], 0x07030602u);
    const unsigned a23 = __builtin_amdgcn_perm(x[3], x[2], 0x05010400u);
    const unsigned b23 = __builtin_amdgcn_perm(x[3], x[2], 0x07030602u);
    out[0] = __builtin_amdgcn_perm(a23, a01, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(a23, a01, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(b23, b01, 0x05040100u);
    out[3] = __builtin_amdgcn_perm(b23, b01, 0x07060302u);
}

template <class Src>
__global__ __launch_bounds__(256) void prep_split_kernel(Src src, int P, int G32,
                                                         const std::int64_t* __restrict__ bt_s0,
                                                         const std::int32_t* __restrict__ bt_len,
                                                         const std::int64_t* __restrict__ bt_k0,
                                                         const std::int32_t* __restrict__ chunk_block,
                                                         std::int64_t n_chunks, std::int64_t KS32,
                                                         std::uint8_t* __restrict__ planes) {
    __shared__ Stage st;
    const int tid = threadIdx.x;
    // thread -> (q or w digits, 32-SNP step of the chunk, fragment lane)
    const int lane = tid & 63, step = (tid >> 6) & 1;
    const int set = __builtin_amdgcn_readfirstlane(tid >> 7);
    const std::int64_t n_units = static_cast<std::int64_t>(G32) * n_chunks;
    // Units run chunk-fastest so consecutive workgroups read adjacent row segments and
    // write adjacent plane chunks.  The next unit's inputs are fetched into registers
    // before the current unit is converted, so their latency overlaps the conversion,
    // and the stage is refilled only after the current unit's stores are issued: each
    // refill then waits for its own loads, never for the plane stores issued after them.
    // The first unit's stage is filled before the loop, and the last iteration re-reads
    // a valid unit, so that every path through the loop issues the same operations.
    std::int64_t u = blockIdx.x;
    if (u >= n_units) return;
    PrepUnit cur = prep_unit(u, n_chunks, bt_s0, bt_len, bt_k0, chunk_block);
    src.put(src.fetch(32 * cur.g, P, cur.snp0, cur.live, tid), tid, st);
    lds_barrier();
    for (;;) {
        const bool more = u + gridDim.x < n_units;
        const PrepUnit nxt = prep_unit(more ? u + gridDim.x : u, n_chunks, bt_s0, bt_len, bt_k0, chunk_block);
        const typename Src::Raw raw = src.fetch(32 * nxt.g, P, nxt.snp0, nxt.live, tid);

        // Digit k of an integer is its byte 5 - k: digits 5..2 come from the low dword,
        // digits 1 and 0 from this set's half of the shared one.
        unsigned pl[kSetPlanes][4];
        const unsigned* lo = set ? st.w : st.q;
        const unsigned sel = set ? 0x07030602u : 0x05010400u;
#pragma unroll
        for (int j4 = 0; j4 < 4; ++j4) {
            const int at = (lane & 31) * kStageLd + 32 * step + 16 * (lane >> 5) + 4 * j4;
            const unsigned x[4] = {lo[at], lo[at + 1], lo[at + 2], lo[at + 3]};
            unsigned by[4];
            bytes4x4(x, by);
#pragma unroll
            for (int i = 0; i < 4; ++i) pl[5 - i][j4] = by[i];
            const unsigned t01 = __builtin_amdgcn_perm(st.t[at + 1], st.t[at], sel);
            const unsigned t23 = __builtin_amdgcn_perm(st.t[at + 3], st.t[at + 2], sel);
            pl[1][j4] = __builtin_amdgcn_perm(t23, t01, 0x05040100u);
            pl[0][j4] = __builtin_amdgcn_perm(t23, t01, 0x07060302u);
        }
        std::uint8_t* base =
            planes + ((static_cast<std::int64_t>(cur.g) * KS32 + 2 * cur.c + step) * kPlanes + kSetPlanes * set) * kChunk +
            lane * 16;
        // Streaming stores: the planes are far larger than the caches and are read back
        // by a later kernel in another order.
#pragma unroll
        for (int p = 0; p < kSetPlanes; ++p)
            __builtin_nontemporal_store(u4v{pl[p][0], pl[p][1], pl[p][2], pl[p][3]},
                                        reinterpret_cast<u4v*>(base + p * kChunk));
        if (!more) break;
        lds_barrier();  // every reader of this unit's stage is done
        src.put(raw, tid, st);
        lds_barrier();
        cur = nxt;
        u += gridDim.x;
    }
}

// ---------------------------------------------------------------------------------
// pair counts: vpair_ij = sum_s v_i v_j by int8 MFMA (exact int32), written for both
// (i,j) and (j,i).  An entry is observed when bit 6 of its byte is set, in fragments of 32
// rows x 32 SNPs `stride` bytes apart (the split form's W_0' plane, or the FP64 form's V
// plane).  Persistent 4-wavefront workgroups over (block, 128x128 tile pair) items;
// wavefront w owns the 64x64 quadrant (rows 64 (w & 1), columns 64 (w >> 1)), so every
// fragment a wavefront loads is loaded by one other wavefront of the workgroup at the same
// time (the second load hits the CU's L1).  Quadrants below the diagonal of a diagonal
// tile pair are skipped.  Two K-steps are in flight while the two before them are
// multiplied (blocks are padded to 64 SNPs, so steps come in pairs).
// ---------------------------------------------------------------------------------
__device__ inline i4 observed(i4 x) { return (x >> 6) & 0x01010101; }

__global__ __launch_bounds__(256) void count_kernel(const std::uint8_t* __restrict__ vplane, std::int64_t stride,
                                                    BlockTable bt, const F2Item* __restrict__ items,
                                                    ItemQueues queues, unsigned* __restrict__ counters, int P,
                                                    int G32, std::int64_t KS32, double* __restrict__ vpair) {
    __shared__ int s_item;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int rh = wave & 1, ch = wave >> 1;
    const std::int64_t slab = static_cast<std::int64_t>(P) * P;
    const int home = static_cast<int>(blockIdx.x % kXcds);
    int xq = 0;
    for (;;) {
        if (threadIdx.x == 0) s_item = claim_item(counters, queues, home, xq);
        __syncthreads();
        const int it = __builtin_amdgcn_readfirstlane(s_item);
        __syncthreads();
        if (it < 0) break;
        const F2Item wi = items[it];
        const int b = __builtin_amdgcn_readfirstlane(wi.b);
        const int ti = __builtin_amdgcn_readfirstlane(static_cast<int>(wi.ti));
        const int tj = __builtin_amdgcn_readfirstlane(static_cast<int>(wi.tj));
        if (ti == tj && rh > ch) continue;
        const int gI0 = 4 * ti + 2 * rh;
        const int gJ0 = 4 * tj + 2 * ch;
        if (gI0 >= G32 || gJ0 >= G32) continue;
        const std::int64_t t0 = bt.k0[b] / 32;
        const int nsteps = __builtin_amdgcn_readfirstlane(bt.kpad[b] / 32);
        // the second group of a pair past the last one re-reads the first (never written out)
        const std::uint8_t* pI[2];
        const std::uint8_t* pJ[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            pI[x] = vplane + (static_cast<std::int64_t>(gI0 + x < G32 ? gI0 + x : gI0) * KS32 + t0) * stride + lane * 16;
            pJ[x] = vplane + (static_cast<std::int64_t>(gJ0 + x < G32 ? gJ0 + x : gJ0) * KS32 + t0) * stride + lane * 16;
        }
        i16v cnt[2][2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) cnt[x][y] = i16v{};
        i4 cI[2][2], cJ[2][2];
        auto load = [&](int t, i4 (&fI)[2][2], i4 (&fJ)[2][2]) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    fI[u][x] = *reinterpret_cast<const i4*>(pI[x] + (t + u) * stride);
                    fJ[u][x] = *reinterpret_cast<const i4*>(pJ[x] + (t + u) * stride);
                }
        };
        if (nsteps > 0) load(0, cI, cJ);
        for (int t = 0; t < nsteps; t += 2) {
            i4 nI[2][2], nJ[2][2];
            load(t + 2 < nsteps ? t + 2 : t, nI, nJ);   // the last pair re-reads itself
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                i4 vI[2], vJ[2];
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    vI[x] = observed(cI[u][x]);
                    vJ[x] = observed(cJ[u][x]);
                }
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 2; ++y)
                        cnt[x][y] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vI[x], vJ[y], cnt[x][y], 0, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    cI[u][x] = nI[u][x];
                    cJ[u][x] = nJ[u][x];
                }
        }
        double* vpb = vpair + slab * b;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const int gI = gI0 + x, gJ = gJ0 + y;
                if (gI >= G32 || gJ >= G32 || gI > gJ) continue;
                const int col = 32 * gJ + (lane & 31);
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int row = 32 * gI + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                    if (row >= P || col >= P || (gI == gJ && row > col)) continue;
                    const double vp = static_cast<double>(cnt[x][y][e]);
                    vpb[row + static_cast<std::int64_t>(P) * col] = vp;
                    vpb[col + static_cast<std::int64_t>(P) * row] = vp;
                }
            }
    }
}

// ---------------------------------------------------------------------------------
// The split contraction.
// ---------------------------------------------------------------------------------
__device__ inline i4 lds_frag(const std::uint8_t* slot, int group, int plane, int lane) {
    return *reinterpret_cast<const i4*>(slot + (group * kSetPlanes + plane) * kChunk + lane * 16);
}

// V = -128 v from W_0': bit 6 of each byte moved to its sign bit.
__device__ inline i4 v_of_w0(i4 w0) {
    u4v x = __builtin_bit_cast(u4v, w0);
    x = (x << 1) & 0x80808080u;
    return __builtin_bit_cast(i4, x);
}

// s_waitcnt on the vector-memory count and, to zero, on this wavefront's LDS reads (gfx9
// encoding: vmcnt in bits 3:0 and 15:14, lgkmcnt 11:8; expcnt 6:4 left at its maximum): at a
// phase barrier no read of the slot that is refilled next may still be under way, wherever
// the compiler put the products that use it.  As a builtin, unlike inline assembly, the
// compiler's wait-count tracking takes it into account.
template <int N>
__device__ inline void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
}

// Issue this wavefront's share of one slot's 1 KB chunks (direct global->LDS): chunk
// ci = wave + 8 r from its source row `src[r]` (uniform) at byte `off` (per lane).
// Every wavefront issues exactly kSetPlanes loads per slot, and chunk ci of a slot is
// always loaded by wavefront ci % 8; the compile-time count lets the compiler's
// wait-count tracking see how many loads follow each slot's, so that it adds no wait of
// its own beyond the explicit ones.
__device__ inline void stage_slot(const std::uint8_t* const (&src)[kSetPlanes], std::uint8_t* slot, unsigned off,
                                  int wave) {
#pragma unroll
    for (int r = 0; r < kSetPlanes; ++r)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[r] + off),
                                         (__attribute__((address_space(3))) void*)(slot + (wave + kWaves * r) * kChunk),
                                         16, 0, 0);
}

// The products of one phase for the wavefront's NX sub-tiles: left groups li .. li + NX - 1
// against right group rj of a slot.  Where the LDS reads stand is the compiler's choice: with
// each left fragment read one product group ahead, extractions of 10 to 1000 populations were
// as fast at best and up to 4% slower.
template <int NX>
__device__ __forceinline__ void mul_q(i16v (&L)[NX][6], const std::uint8_t* slot, int li, int rj, int lane) {
    i4 dj[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) dj[k] = lds_frag(slot, rj, k, lane);
    static_for<6>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            const i4 di = lds_frag(slot, li + x, k, lane);
#pragma unroll
            for (int t = k; t < 6; ++t)
                L[x][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(di, dj[t - k], L[x][t], 0, 0, 0);
        }
    });
}

template <int NX>
__device__ __forceinline__ void mul_w(i16v (&L)[NX][6], const std::uint8_t* slot, int li, int rj, int lane) {
    i4 wj[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) wj[k] = lds_frag(slot, rj, k, lane);
    const i4 vj = v_of_w0(wj[0]);
#pragma unroll
    for (int x = 0; x < NX; ++x) {
        const i4 w0 = lds_frag(slot, li + x, 0, lane);
        const i4 vi = v_of_w0(w0);
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            const i4 wt = t == 0 ? w0 : lds_frag(slot, li + x, t, lane);
            L[x][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wt, vj, L[x][t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 6; ++t) L[x][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vi, wj[t], L[x][t], 0, 0, 0);
    }
}

// One work item as a wavefront sees it (every field uniform): a block's K range, the tile's
// row groups, and the wavefront's NX sub-tiles, left groups gI .. gI + NX - 1 (li in the
// slot) against right group gJ (rj in the slot).
struct WaveItem {
    std::int64_t t0;          // the block's first K-step
    int b, nsteps;
    int gI0, gJ0;             // the workgroup tile's first left and right row group
    int gI, gJ, li, rj;
};

// Every wavefront of the workgroup runs the same number of barriers whatever its NX.
template <int NX>
__device__ __forceinline__ void run_item(const WaveItem& wi, const std::uint8_t* __restrict__ planes,
                                         std::int64_t KS32, int G32, int P, const double* __restrict__ vpair,
                                         double* __restrict__ f2, const FixupList& fl, std::uint8_t* lds_0,
                                         std::uint8_t* lds_1, std::uint8_t* lds_2, int wave, int lane) {
    const int nsteps = wi.nsteps;
    const std::int64_t slab = static_cast<std::int64_t>(P) * P;
    for (int seg0 = 0;; seg0 += kSegSteps) {
        const int seg_end = nsteps < seg0 + kSegSteps ? nsteps : seg0 + kSegSteps;
        const bool last_seg = seg_end == nsteps;
        const std::uint8_t* src[kSetPlanes];
#pragma unroll
        for (int r = 0; r < kSetPlanes; ++r) {
            const int ci = wave + kWaves * r;
            const int lg = ci / kSetPlanes, pp = ci - lg * kSetPlanes;
            int gg = lg < 4 ? wi.gI0 + lg : wi.gJ0 + lg - 4;
            if (gg >= G32) gg = 0;  // rows beyond P: any valid address; never read back
            src[r] = planes + ((static_cast<std::int64_t>(gg) * KS32 + wi.t0 + seg0) * kPlanes + pp) * kChunk;
        }
        // Byte offset of plane set `set` of step s (look-ahead past the segment's end
        // re-reads its last K-step, an empty block's prologue the step it was given; neither
        // is read back).
        auto offset = [&](int s, int set) {
            const int k = s < seg_end ? s - seg0 : (seg_end > seg0 ? seg_end - 1 - seg0 : 0);
            return static_cast<unsigned>((k * kPlanes + kSetPlanes * set) * kChunk + lane * 16);
        };
        i16v L[NX > 0 ? NX : 1][6];
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
            for (int t = 0; t < 6; ++t) L[x][t] = i16v{};

        // Phase p = 2 step + set reads slot p % 3.  Per wavefront six loads per slot, all
        // unconditional, so the explicit waits are exact on every path:
        //   prologue:  D(0) -> slot 0, W(0) -> slot 1
        //   phase p:   wait until at most six loads (phase p + 1's) are outstanding, so
        //              this phase's have landed; barrier (every wavefront's have, and
        //              every reader of phase p - 1's slot is done); issue phase p + 2
        //              into that slot; multiply.
        auto step_body = [&]<int r>(int step) {
            std::uint8_t* const slots[3] = {lds_0, lds_1, lds_2};
            constexpr int pd = (2 * r) % 3, pw = (2 * r + 1) % 3, pf = (2 * r + 2) % 3;
            wait_vmcnt<kSetPlanes>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            stage_slot(src, slots[pf], offset(step + 1, 0), wave);
            if constexpr (NX > 0) mul_q<NX>(L, slots[pd], wi.li, wi.rj, lane);
            wait_vmcnt<kSetPlanes>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            stage_slot(src, slots[pd], offset(step + 1, 1), wave);
            if constexpr (NX > 0) mul_w<NX>(L, slots[pw], wi.li, wi.rj, lane);
        };
        if (seg0 > 0) __syncthreads();  // every reader of the previous segment's slots is done
        stage_slot(src, lds_0, offset(seg0, 0), wave);
        stage_slot(src, lds_1, offset(seg0, 1), wave);
        // The slot pattern repeats every three steps, so that each slot is a distinct LDS
        // object in every access.
        int step = seg0;
        for (; step + 2 < seg_end; step += 3) {
            step_body.template operator()<0>(step);
            step_body.template operator()<1>(step + 1);
            step_body.template operator()<2>(step + 2);
        }
        if (step < seg_end) step_body.template operator()<0>(step);
        if (step + 1 < seg_end) step_body.template operator()<1>(step + 1);

        // Epilogue: num = -2 sum_t U_t L_t; f2 = num / vpair.  The three upper and the
        // three lower levels are combined exactly in 64-bit integers.  W_0's offset is
        // taken back with the pairs counted up to each segment's end (for a segment before
        // the last an integer share of them: the shares add up to the count).
        double* f2b = f2 + slab * wi.b;
        const double* vpb = vpair + slab * wi.b;
        int el = lane;
        asm volatile("" : "+v"(el));  // the output addresses are formed here, not kept through the K loop
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            const int gI = wi.gI + x;
            const int col = 32 * wi.gJ + (el & 31);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = 32 * gI + 8 * (e >> 2) + 4 * (el >> 5) + (e & 3);
                const bool ok = row < P && col < P && !(gI == wi.gJ && row > col);
                double val = 0.0, vp = 0.0;
                if (ok) {
                    const std::int64_t ij = row + static_cast<std::int64_t>(P) * col;
                    vp = vpb[ij];
                    int share = static_cast<int>(vp);
                    if (seg0 > 0 || !last_seg) {
                        const std::int64_t pairs = share;
                        share = static_cast<int>(pairs * seg_end / nsteps) - static_cast<int>(pairs * seg0 / nsteps);
                    }
                    const std::int64_t l0 = L[x][0][e] + static_cast<std::int64_t>(kL0PerPair) * share;
                    const std::int64_t hi = (l0 << 16) + (static_cast<std::int64_t>(L[x][1][e]) << 8) + L[x][2][e];
                    const std::int64_t lo = (static_cast<std::int64_t>(L[x][3][e]) << 16) +
                                            (static_cast<std::int64_t>(L[x][4][e]) << 8) + L[x][5][e];
                    double num = -2.0 * (static_cast<double>(hi) * 0x1p-30 + static_cast<double>(lo) * 0x1p-54);
                    if (seg0 > 0) num += f2b[ij];
                    val = last_seg ? (vp > 0.0 ? num / vp : 0.0) : num;
                    f2b[ij] = val;
                    if (last_seg) f2b[col + static_cast<std::int64_t>(P) * row] = val;
                }
                if (last_seg) fixup_append(fl, ok && vp > 0.0 && fabs(val) < fl.tau, wi.b, row, col);
            }
        }
        if (last_seg) break;
    }
}

__global__ __launch_bounds__(512) void f2_split_kernel(const std::uint8_t* __restrict__ planes, BlockTable bt,
                                                       const F2Item* __restrict__ items, ItemQueues queues,
                                                       unsigned* __restrict__ counters, int P, int G32,
                                                       std::int64_t KS32, const double* __restrict__ vpair,
                                                       double* __restrict__ f2, FixupList fl) {
    // One LDS object per ring slot: the compiler then knows that reads of one slot do
    // not depend on the direct loads still landing in the others.
    __shared__ __attribute__((aligned(16))) std::uint8_t lds_0[kSlotBytes];
    __shared__ __attribute__((aligned(16))) std::uint8_t lds_1[kSlotBytes];
    __shared__ __attribute__((aligned(16))) std::uint8_t lds_2[kSlotBytes];
    __shared__ int s_item;
    const int lane = threadIdx.x & 63;
    // Wavefront-uniform values are moved to scalar registers so that every branch
    // on them is uniform and the MFMA accumulators never sit in divergent flow.
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));

    const int home = static_cast<int>(blockIdx.x % kXcds);
    int xq = 0;
    for (;;) {
        if (threadIdx.x == 0) s_item = claim_item(counters, queues, home, xq);
        __syncthreads();
        const int it = __builtin_amdgcn_readfirstlane(s_item);
        __syncthreads();
        if (it < 0) break;
        const F2Item f = items[it];
        WaveItem wi;
        wi.b = __builtin_amdgcn_readfirstlane(f.b);
        wi.gI0 = 4 * __builtin_amdgcn_readfirstlane(static_cast<int>(f.ti));
        wi.gJ0 = 4 * __builtin_amdgcn_readfirstlane(static_cast<int>(f.tj));
        wi.t0 = bt.k0[wi.b] / 32;
        if (wi.t0 >= KS32) wi.t0 = KS32 > 0 ? KS32 - 1 : 0;  // an empty last block: any valid step
        wi.nsteps = __builtin_amdgcn_readfirstlane(bt.kpad[wi.b] / 32);

        // This wavefront's 32x32 sub-tiles: left groups li and li + 1, right group wc.
        // Off the diagonal two row pairs x four columns.  A diagonal tile has the ten
        // sub-tiles with li <= wc, dealt so that no SIMD (wavefronts w and w + 4) has more
        // than three: (0,1) (1,1) | (0,2) (1,2) | (0,3) (1,3) | (2,3) (3,3) | (0,0) | (2,2).
        const bool diag = wi.gI0 == wi.gJ0;
        wi.li = diag ? 2 * ((0xE8 >> wave) & 1) : 2 * (wave & 1);
        const int wc = diag ? (0x00203321 >> (4 * wave)) & 15 : wave >> 1;
        wi.rj = 4 + wc;
        wi.gI = wi.gI0 + wi.li;
        wi.gJ = wi.gJ0 + wc;
        int n_act = 0;
#pragma unroll
        for (int x = 0; x < 2; ++x)
            n_act += wi.gI + x < G32 && wi.gJ < G32 && (!diag || wi.li + x <= wc);
        if (n_act == 2) run_item<2>(wi, planes, KS32, G32, P, vpair, f2, fl, lds_0, lds_1, lds_2, wave, lane);
        else if (n_act == 1) run_item<1>(wi, planes, KS32, G32, P, vpair, f2, fl, lds_0, lds_1, lds_2, wave, lane);
        else run_item<0>(wi, planes, KS32, G32, P, vpair, f2, fl, lds_0, lds_1, lds_2, wave, lane);
    }
    // The last item's look-ahead loads may still be landing in LDS: drain them before
    // the workgroup's LDS can be handed to another workgroup.
    wait_vmcnt<0>();
}

}  // namespace

// Persistent-style grid for the prep: enough workgroups to fill every CU several
// times over, each looping over (32-row group, chunk) units.
static unsigned prep_grid(std::int64_t n_units) {
    return static_cast<unsigned>(std::max<std::int64_t>(1, std::min<std::int64_t>(n_units, 8192)));
}

void launch_prep_split_counts(const std::uint16_t* a2, const std::uint16_t* n, std::int64_t ld, int P, int G32,
                              BlockTable bt, const std::int32_t* chunk_block, std::int64_t n_chunks,
                              std::int64_t KS32, std::uint8_t* planes, hipStream_t st) {
    if (n_chunks <= 0 || G32 <= 0) return;
    prep_split_kernel<CountsSrc><<<prep_grid(G32 * n_chunks), 256, 0, st>>>(
        CountsSrc{a2, n, ld}, P, G32, bt.s0, bt.len, bt.k0, chunk_block, n_chunks, KS32, planes);
    STP_LAUNCH_CHECK();
}

void launch_prep_split_qvn(const double* q, const double* v, const double* n, int P, int G32, BlockTable bt,
                           const std::int32_t* chunk_block, std::int64_t n_chunks, std::int64_t KS32,
                           std::uint8_t* planes, hipStream_t st) {
    if (n_chunks <= 0 || G32 <= 0) return;
    prep_split_kernel<QvnSrc><<<prep_grid(G32 * n_chunks), 256, 0, st>>>(
        QvnSrc{q, v, n}, P, G32, bt.s0, bt.len, bt.k0, chunk_block, n_chunks, KS32, planes);
    STP_LAUNCH_CHECK();
}

void launch_count_split(const std::uint8_t* planes, BlockTable bt, const F2Item* items, const ItemQueues& queues,
                        unsigned* counters, int P, int G32, std::int64_t KS32, double* vpair, int n_workgroups,
                        hipStream_t st) {
    if (queues.off[kXcds] <= 0) return;
    launch_zero_u32(counters, kXcds, st);
    count_kernel<<<static_cast<unsigned>(n_workgroups), 256, 0, st>>>(
        planes + kSetPlanes * kChunk, kPlanes * kChunk, bt, items, queues, counters, P, G32, KS32, vpair);
    STP_LAUNCH_CHECK();
}

void launch_count_v8(const std::uint8_t* v8, BlockTable bt, const F2Item* items, const ItemQueues& queues,
                     unsigned* counters, int P, int G32, std::int64_t KS32, double* vpair, int n_workgroups,
                     hipStream_t st) {
    if (queues.off[kXcds] <= 0) return;
    launch_zero_u32(counters, kXcds, st);
    count_kernel<<<static_cast<unsigned>(n_workgroups), 256, 0, st>>>(v8, kChunk, bt, items, queues, counters, P, G32,
                                                                      KS32, vpair);
    STP_LAUNCH_CHECK();
}

void launch_f2_split(const std::uint8_t* planes, BlockTable bt, const F2Item* items, const ItemQueues& queues,
                     unsigned* counters, int P, int G32, std::int64_t KS32, const double* vpair, double* f2,
                     const FixupList& fl, int n_workgroups, hipStream_t st) {
    if (queues.off[kXcds] <= 0) return;
    launch_zero_u32(counters, kXcds, st);
    f2_split_kernel<<<static_cast<unsigned>(n_workgroups), 512, 0, st>>>(planes, bt, items, queues, counters, P, G32,
                                                                         KS32, vpair, f2, fl);
    STP_LAUNCH_CHECK();
}

}  // namespace stp
