// Producer GEMM: C[M,N] = A[M,K] . Bt[N,K]^T (+ bias[N]) on CDNA4 MFMA.
//
// Replaces the reference's aclnnMatmul producer (exec/qwen_main.cpp:499-512,
// exec/runtime/op_impl.cpp:175-201). Weights are re-laid out once at load as
// Bt = weight_t^T ([N,K], K contiguous) so that both operands feed the MFMA
// with one 16-byte load per lane.
//
// * 4 waves in a 2x2 grid (each wave owns (BM/2)x(BN/2) of C), or for
//   256x256 tiles 8 waves in a 2x4 grid (128x64 each, two waves per SIMD), as
//   32x32 accumulator blocks (fp32). The 8-wave register-staged kernels and
//   the simple kernel compute a block as four 16x16 sub-blocks with
//   v_mfma_f32_16x16x32 (4 values per lane each), and so does the 4-wave wide
//   loop of the 256-wide tiles with long K; the other 4-wave direct-to-LDS
//   kernels as one block with v_mfma_f32_32x32x16 (16 values per lane). The
//   16x16x32 instruction reads and writes a quarter of the accumulator
//   registers of 32x32x16 per flop; under the card's power limit an
//   MFMA-only loop of it held 2.31 GHz against 1.95-2.10 GHz at the same
//   busy fraction (kernrelay_amd/probes/mfma_power.hip).
// * K is walked in 64-wide steps through a double-buffered LDS stage; global
//   loads of step k+1 are in flight while step k runs on the matrix cores.
// * LDS rows are 128 B (64 elements); the 16-byte chunk index is XOR-swizzled
//   with (row>>1)&7, under which the 16 lanes of a fragment read (16
//   consecutive rows, one chunk) hit distinct banks (0 conflict cycles
//   measured by kernrelay_amd/probes/lds_banks.hip).
// * Every data-parallel variant walks K in the same order, and the two MFMA
//   shapes give the same bits for the same K order, so a row of C is
//   bit-identical whatever BM/BN or row range a launch covers: the split
//   schedule is bit-exact against the unsplit one. The split-K kernels
//   (stream-K, GemmSplitKernel) sum their pieces of K in piece order: their bits
//   follow the plan, a function of M, N and K alone, and differ from the
//   data-parallel ones by the order of the fp32 sums.
// * The MFMA is fed (B fragment, A fragment), so each block holds C^T: in a
//   16x16 sub-block lane l owns row l % 16 and columns 4 (l / 16) .. + 3, in
//   a 32x32 block row l % 32 and four runs of 4 columns.
// * Epilogue: acc -> 16-bit (RNE); with bias, bf16(bf16(acc)+bias) — the
//   rounding of the reference's separate Matmul then Add (EmitQkv,
//   exec/qwen_main.cpp:1336-1344). The tile is staged row-major in LDS
//   (8-byte writes, XOR-swizzled) and leaves as full-line 16-byte stores. Then
//   the workgroup arrives on its row tile's relay counter; the last arrival
//   releases the tile.
#include "kr_dma.h"
#include "kr_gemm.h"
#include "kr_relay.h"
#include "kr_rowcore.h"
#include "kr_rowops.h"

namespace kr {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kBK = 64;          // K elements per LDS stage
constexpr int kRowChunks = 8;    // 16-byte chunks per LDS row
constexpr int kThreads = 256;

struct GemmParams {
    const uint16_t *A;
    const uint16_t *Bt;
    uint16_t *C;
    const uint16_t *bias;
    int64_t lda, ldb, ldc;
    int M, N, K;
    int tiles_m, tiles_n;
    int order_rows;  // > 0: dispatch tiles in relay-tile order, this many rows each
    int group_m;     // raster: row blocks per group (0 = all)
    int store_kind;  // 0 device-scope (default), 1 plain, 2 nontemporal
    RelayPub pub;
    RelayWait wait;
    uint16_t *tail_act;  // SwiGLU tail consumer output (nullptr: none)
    int tail_cols;
    uint16_t *epi_act;   // SwiGLU epilogue output [M, N/2] (nullptr: store C)
    int64_t ld_act;
    void *uy;        // unary consumer output (nullptr: none)
    int uop, udt;
    int64_t ldy;
    int sk_wgs;          // stream-K workgroups (0: one tile per workgroup)
    int sk_pmax;         // partial-sum slots per tile in sk_ws
    float *sk_ws;        // [tiles][sk_pmax][BM*BN] fp32 partials
    int32_t *sk_cnt;     // [tiles] arrival counters, zero between launches
    int gemm_wgs;        // workgroups of the GEMM proper; the rest are tail
    int tail_wpt;        // tail workgroups per relay tile
    const uint16_t *rope_cos;  // RoPE epilogue (nullptr: none)
    const uint16_t *rope_sin;
    int rope_cols, rope_d, rope_pos0;
    // Add+RMSNorm relay consumer run by the producer's workgroups (rn_y ==
    // nullptr: none): y = rmsnorm(res + C) * gamma, sum = res + C, per row of
    // every released relay tile; all [M, N] packed
    const uint16_t *rn_res;
    const uint16_t *rn_gamma;
    uint16_t *rn_y;
    uint16_t *rn_sum;
    float *rn_rstd;
    float rn_eps;
    int rn_cpl;          // chunks per lane of a one-wave row (1, 2, 4, 8)
    uint32_t rn_spins;   // spin bound of the wait on a relay tile
};

__device__ __forceinline__ int Swz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// Workgroup -> output tile. The dispatcher deals workgroups to the 8 XCDs
// round-robin (XCD = blockIdx % 8) and each XCD has its own L2. Within a run
// of `per` consecutive workgroup ids starting at `first`, XCD x takes a
// contiguous chunk of the run's tiles, so a weight column block is read by
// workgroups of one XCD while it sits in that XCD's L2.
// * No relay: one run over all tiles, rastered in groups of group_m row
//   blocks (row blocks fastest within a group), so the tiles an XCD runs at
//   once form a near-square patch of C.
// * Relay (order_rows > 0): one run per relay tile, front to back, so tile 0
//   of the rows is complete first; each run covers order_rows/bm row blocks,
//   odd runs with the weight columns in reverse (each run reads all of the
//   weight, and the blocks the last run read are the ones still cached).

__device__ __forceinline__ void TileOf(int bid, int tiles_m, int tiles_n, int bm, int order_rows, int group_m, int &tm,
                                       int &tn, bool xcd = true)
{
    if (order_rows > 0) {
        const int mt = order_rows / bm;  // row blocks per relay tile
        const int per = mt * tiles_n;
        const int r = bid / per;
        const int t = XcdChunk(bid, r * per, per);
        tm = r * mt + t % mt;
        tn = t / mt;
        // serpentine: odd relay tiles walk the weight columns backwards, so
        // they start on the blocks the previous tile read last (still in MALL)
        if (r & 1) tn = tiles_n - 1 - tn;
        return;
    }
    // grouped raster: runs of `group_m` row blocks fastest, so an XCD's
    // concurrent tiles form a near-square patch (fewer distinct operand
    // slices per K stage in its L2) rather than a tall column
    const int t = xcd ? XcdChunk(bid, 0, tiles_m * tiles_n) : bid;
    const int gm_all = group_m > 0 ? min(group_m, tiles_m) : tiles_m;
    const int per_group = gm_all * tiles_n;
    const int g = t / per_group;
    const int first_m = g * gm_all;
    const int gm = min(tiles_m - first_m, gm_all);
    const int r = t - g * per_group;
    tm = first_m + r % gm;
    tn = r / gm;
}

// One 16x16x32 MFMA on a 16x16 sub-block: a holds 16 rows of the A operand
// (lane l: row l % 16, k 8 (l / 16) .. + 7), b 16 columns of the B operand
// likewise; c: lane l holds column l % 16, rows 4 (l / 16) .. + 3.
template <int DT>
__device__ __forceinline__ f32x4 Mfma(const uint4 &a, const uint4 &b, const f32x4 &c)
{
    if constexpr (DT == kBF16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
}

// One 32x32x16 MFMA on a whole 32x32 block (the direct-to-LDS loop of the
// 4-wave kernels, which measured faster with it): a and b hold 32 rows of
// their operand (lane l: row l % 32, k 8 (l / 32) .. + 7); c: lane l holds
// column l % 32, rows 8 (v / 4) + 4 (l / 32) + v % 4. For the same K order
// it gives the same bits as four 16x16x32 MFMAs over the block's quarters
// (the 7B prefill's logits hash is equal with either).
template <int DT>
__device__ __forceinline__ f32x16 Mfma32(const uint4 &a, const uint4 &b, const f32x16 &c)
{
    if constexpr (DT == kBF16) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
}

// Accumulator helpers over both layouts: block (i, j), four-value group c,
// value e (the order stream-K partials are written and read back in).
template <int MI, int NI>
__device__ __forceinline__ void AccZero(f32x4 (&a)[MI][NI][4])
{
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) a[i][j][q][e] = 0.0f;
}
template <int MI, int NI>
__device__ __forceinline__ void AccZero(f32x16 (&a)[MI][NI])
{
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) a[i][j][e] = 0.0f;
}
template <int MI, int NI>
__device__ __forceinline__ float AccAt(const f32x4 (&a)[MI][NI][4], int i, int j, int c, int e)
{
    return a[i][j][c][e];
}
template <int MI, int NI>
__device__ __forceinline__ float AccAt(const f32x16 (&a)[MI][NI], int i, int j, int c, int e)
{
    return a[i][j][4 * c + e];
}
template <int MI, int NI>
__device__ __forceinline__ void AccSet(f32x4 (&a)[MI][NI][4], int i, int j, int c, int e, float v)
{
    a[i][j][c][e] = v;
}
template <int MI, int NI>
__device__ __forceinline__ void AccSet(f32x16 (&a)[MI][NI], int i, int j, int c, int e, float v)
{
    a[i][j][4 * c + e] = v;
}

// ---------------------------------------------------------------- tail
// Gate/up halves of four output chunks of an interleaved gate/up buffer
// (chunk c: 8 gate then 8 up values at c*16), all eight loads device-scope
// (the tile was released by other XCDs' device-scope stores; this XCD's L2
// may hold stale lines of the buffer from an earlier use) and in flight
// together; returns once they have landed.
typedef uint32_t GemmU32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void LoadGateUp4(const uint16_t *p0, const uint16_t *p1, const uint16_t *p2,
                                            const uint16_t *p3, GemmU32x4 (&g)[4], GemmU32x4 (&u)[4])
{
    asm volatile(
        "global_load_dwordx4 %0, %8, off sc1\n\t"
        "global_load_dwordx4 %1, %8, off offset:16 sc1\n\t"
        "global_load_dwordx4 %2, %9, off sc1\n\t"
        "global_load_dwordx4 %3, %9, off offset:16 sc1\n\t"
        "global_load_dwordx4 %4, %10, off sc1\n\t"
        "global_load_dwordx4 %5, %10, off offset:16 sc1\n\t"
        "global_load_dwordx4 %6, %11, off sc1\n\t"
        "global_load_dwordx4 %7, %11, off offset:16 sc1\n\t"
        "s_waitcnt vmcnt(0)"
        : "=&v"(g[0]), "=&v"(u[0]), "=&v"(g[1]), "=&v"(u[1]), "=&v"(g[2]), "=&v"(u[2]), "=&v"(g[3]), "=&v"(u[3])
        : "v"(p0), "v"(p1), "v"(p2), "v"(p3)
        : "memory");
}

// SwiGLU of one chunk, rounded exactly as the standalone kernel rounds it:
// the silu result is stored (16-bit) before the multiply.
template <int DT>
__device__ __forceinline__ uint4 SwigluChunk(const GemmU32x4 &g, const GemmU32x4 &u)
{
    U16x8 a, b, r;
    *reinterpret_cast<GemmU32x4 *>(a.v) = g;
    *reinterpret_cast<GemmU32x4 *>(b.v) = u;
#pragma unroll
    for (int e = 0; e < 8; ++e)
        r.v[e] = Elem<DT>::Store(RoundTo<DT>(Silu(Elem<DT>::Load(a.v[e]))) * Elem<DT>::Load(b.v[e]));
    return *reinterpret_cast<const uint4 *>(r.v);
}

// A tail workgroup: wait for its relay tile, SwiGLU over its share of the
// tile's rows; the last one of the tile consumes the release.
template <int DT>
__device__ void TailSwiglu(const GemmParams &p)
{
    const int j = int(blockIdx.x) - p.gemm_wgs;
    const int t = j / p.tail_wpt;
    const int w = j - t * p.tail_wpt;
    int32_t *flag = p.pub.ctrl + size_t(p.pub.flag0 + t) * kWords;
    if (threadIdx.x == 0) SpinOnTile(flag, flag, kDefaultMaxSpins);
    __syncthreads();
    const int64_t rows = p.pub.rows_per_tile;
    const int64_t chunks = rows * p.tail_cols / 8;
    const uint16_t *src = p.C + int64_t(t) * rows * p.ldc;
    uint16_t *dst = p.tail_act + int64_t(t) * rows * p.tail_cols;
    const int64_t stride = int64_t(p.tail_wpt) * blockDim.x;
    int64_t c = int64_t(w) * blockDim.x + threadIdx.x;
    for (; c + 3 * stride < chunks; c += 4 * stride) {
        GemmU32x4 g[4], u[4];
        LoadGateUp4(src + c * 16, src + (c + stride) * 16, src + (c + 2 * stride) * 16, src + (c + 3 * stride) * 16, g,
                    u);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<uint4 *>(dst + (c + q * stride) * 8) = SwigluChunk<DT>(g[q], u[q]);
    }
    for (; c < chunks; c += stride) {
        GemmU32x4 g[4], u[4];
        LoadGateUp4(src + c * 16, src + c * 16, src + c * 16, src + c * 16, g, u);
        *reinterpret_cast<uint4 *>(dst + c * 8) = SwigluChunk<DT>(g[0], u[0]);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int32_t a = __hip_atomic_fetch_add(flag + kOffDone, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a == p.tail_wpt - 1) {
            StoreRelaxed(flag + kOffDone, 0);
            const int32_t to = __hip_atomic_exchange(flag + kOffTimedOut, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            StoreRelaxed(flag + kOffConsumed, LoadRelaxed(flag + kOffConsumed) + 1);
            StoreRelaxed(flag + kOffStatus, to ? 2 : 1);
        }
    }
}

// Finishers that release relay tile r of a split grid: of the row blocks that
// touch it, in every column.
__device__ __forceinline__ int RowTileArrivals(const GemmParams &p, int r, int bm)
{
    const int R = p.pub.rows_per_tile;
    return ((min(r * R + R, p.M) - 1) / bm - r * R / bm + 1) * p.tiles_n;
}

// A split tile's finisher arrives on every relay tile that its rows m0 ..
// m0 + bm - 1 touch. With `place`, LDS ints: its place in the arrival order of
// the i-th goes to place[i].
__device__ __forceinline__ void ArriveRows(const GemmParams &p, int m0, int bm, int *place = nullptr)
{
    if (p.pub.ctrl == nullptr) return;
    RelayPub pub = p.pub;
    const int R = pub.rows_per_tile, r0 = m0 / R;
    for (int r = r0; r * R < min(m0 + bm, p.M); ++r) {
        pub.arrivals = RowTileArrivals(p, r, bm);
        const int a = RelayArrive(pub, r);
        if (place != nullptr && threadIdx.x == 0) place[r - r0] = a;
    }
}

// ------------------------------------------- Add+RMSNorm relay consumer
// The producer's own workgroups consume its released row tiles (the
// reference's down -> Add+RMSNorm tile loop, exec/qwen_main.cpp:1274-1302,
// without the all-reduce): a workgroup that has stored its C tile and arrived
// on the relay tile that its rows are in waits for the tile's release and then
// computes Add+RMSNorm for its share of the tile's rows: as the s-th of
// `workers` arrivals, rows lo + s*waves + wave, stepping by workers*waves, one
// row per wave, RB rows' loads in flight at a time, with the row code of the
// standalone row kernel. C is read at device scope (written by other XCDs'
// workgroups of this launch). The last of the tile's `workers` consumes the
// release (consumed + 1, status 1, or 2 when a wait ran past its spin bound).
//
// A workgroup that waits holds a CU that one of the tile's producers may need:
// another such launch, or anything else on the device, can keep some of them
// from being placed. So a wait ends after kNormPatience at the latest
// without the release: the workgroups leave in the order in which they
// arrived, and the one that releases the tile, which never waits, works the
// shares of those that left after its own. Every placed workgroup ends by
// itself, whatever else runs.
template <int DT, int CPL, int RB>
__device__ __forceinline__ void NormRows(const GemmParams &p, int lo, int hi, int first, int step)
{
    const int ln = threadIdx.x & 63;
    // a wave's rows are the same for all its lanes: kept in scalar registers,
    // the device-scope loads take their base as a plain buffer resource
    // (a row index the compiler thinks may differ per lane would wrap every
    // load in a loop over the lanes' distinct bases)
    first = __builtin_amdgcn_readfirstlane(first);
    if (lo + first >= hi) return;
    uint4 g[CPL];
    RowGammaLoad<CPL>(p.rn_gamma, p.N, ln, g);
    for (int r0 = lo + first; r0 < hi; r0 += RB * step) {
        RowIn<CPL> in[RB];
#pragma unroll
        for (int j = 0; j < RB; ++j) {
            const int r = min(r0 + j * step, hi - 1);  // past the end: re-read, never used
            AddRmsNormLoad<CPL, true>(p.rn_res + int64_t(r) * p.N, p.C + int64_t(r) * p.N, p.N, ln, in[j]);
        }
#pragma unroll
        for (int j = 0; j < RB; ++j) {
            const int r = r0 + j * step;
            if (r >= hi) break;
            const int64_t o = int64_t(r) * p.N;
            AddRmsNormFinish<DT, CPL>(in[j], g, p.rn_y + o, p.rn_sum != nullptr ? p.rn_sum + o : nullptr,
                                      p.rn_rstd != nullptr ? p.rn_rstd + r : nullptr, p.N, p.rn_eps, ln, false);
        }
    }
}

// Spins (about 1 us each) after which a waiting workgroup leaves. The waits of
// a grid that is placed as a whole are shorter: the last pieces' fix-up and
// rows of C, tens of us.
constexpr uint32_t kNormPatience = 512;
constexpr int32_t kLeftReleased = INT32_MIN;  // set in the `left` word by the release

// One lane: wait for the tile as its `place`-th arrival. False: it left.
__device__ __forceinline__ bool NormWait(int32_t *flag, int place, uint32_t max_spins)
{
    const int32_t target = LoadRelaxed(flag + kOffConsumed) + 1;
    uint32_t spins = 0;
    while (LoadRelaxed(flag + kOffPublished) < target) {
        if (++spins > min(max_spins, kNormPatience)) {
            if (spins > max_spins) StoreRelaxed(flag + kOffTimedOut, 1);
            int32_t left = place;  // all earlier ones have left, and the tile is not released
            if (__hip_atomic_compare_exchange_strong(flag + kOffLeft, &left, place + 1, __ATOMIC_RELAXED,
                                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                return false;
        }
        __builtin_amdgcn_s_sleep(2);
    }
    return true;
}

// The part of the `place`-th arrival (thread 0 knows it) of relay tile
// `tile`'s `workers`. slot: two LDS ints. NARROW: rows of up to two chunks per
// lane in flight per wave.
template <int DT, int NW, int WPE, int NARROW = WPE == 2 ? 4 : 8>
__device__ __forceinline__ void NormTail(const GemmParams &p, int tile, int workers, int place, int *slot)
{
    int32_t *flag = p.pub.ctrl + size_t(p.pub.flag0 + tile) * kWords;
    if (threadIdx.x == 0) {
        // (the last arrival released the tile)
        if (place < workers - 1 && !NormWait(flag, place, p.rn_spins)) place = -1;
        slot[0] = place;
    }
    __syncthreads();
    const int R = p.pub.rows_per_tile;
    const int lo = tile * R, hi = min(lo + R, p.M);
    const int step = workers * NW;
    // rows in flight per wave: what the registers hold without spilling
    // (WPE waves per SIMD share its 512 registers; loads land in the 256
    // architectural ones)
    constexpr int CH = WPE == 2 ? 8 : 16;
    int taken = 0;  // thread 0: shares left to this workgroup (known by the end of its own)
    if (threadIdx.x == 0 && place == workers - 1)
        taken = __hip_atomic_fetch_or(flag + kOffLeft, kLeftReleased, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // its own share (none: it left), then shares 0 .. taken - 1
    int i = -1;
    do {
        const int share = i < 0 ? slot[0] : i;
        const int first = share * NW + int(threadIdx.x >> 6);
        if (share >= 0) {
            switch (p.rn_cpl) {
                case 1: NormRows<DT, 1, NARROW>(p, lo, hi, first, step); break;
                case 2: NormRows<DT, 2, NARROW>(p, lo, hi, first, step); break;
                case 4: NormRows<DT, 4, CH / 4>(p, lo, hi, first, step); break;
                default: NormRows<DT, 8, CH / 8>(p, lo, hi, first, step); break;
            }
        }
        if (threadIdx.x == 0) slot[1] = taken;
        __syncthreads();
    } while (++i < slot[1]);
    if (threadIdx.x == 0) {
        const int32_t a = __hip_atomic_fetch_add(flag + kOffDone, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a == workers - 1) {
            StoreRelaxed(flag + kOffDone, 0);
            StoreRelaxed(flag + kOffLeft, 0);
            const int32_t to = __hip_atomic_exchange(flag + kOffTimedOut, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            StoreRelaxed(flag + kOffConsumed, LoadRelaxed(flag + kOffConsumed) + 1);
            StoreRelaxed(flag + kOffStatus, to ? 2 : 1);
        }
    }
}

// The Add+RMSNorm relay consumer of a split tile's finisher, on every relay
// tile that its rows touch. The other pieces' workgroups are done: the
// finishers have a wave for every row of 64 and 128 row tiles, and two to eight
// rows a wave in 256x256 ones (2048x3584x18944 in four relay tiles 251 ->
// 255 us against all pieces on the rows, 2048x896x4864 56 -> 61).
// NARROW 2: with more rows in flight the 256x256 split kernel spills. place: as
// ArriveRows left it. (All workgroups on every relay tile in turn: 768x4096x4096
// in four relay tiles 65 us, 768x3584x18944 155.)
template <int DT, int NW, int WPE>
__device__ __forceinline__ void NormTailRows(const GemmParams &p, int m0, int bm, const int *place, int *slot)
{
    const int R = p.pub.rows_per_tile, r0 = m0 / R;
    for (int r = r0; r * R < min(m0 + bm, p.M); ++r)
        NormTail<DT, NW, WPE, 2>(p, r, RowTileArrivals(p, r, bm), place[r - r0], slot);
}

// The unary consumer's pass over the staged tile (after C's): y = f(C) with
// the elementwise kernel's arithmetic on C's stored values, so y equals what
// that kernel computes from C bit for bit. Every thread stores 16 bytes of y
// per step -- 8 values of a 16-bit y, 4 of an fp32 y -- so each store
// instruction covers whole 128-byte lines (two 16-byte halves of 32-byte
// runs would leave every line half-written per instruction). Staged chunk c
// of a row sits in slot c ^ ((row & 31) >> 1), its 8-byte halves swapped on
// odd rows. Columns past N are not written.
template <int DT, int BM, int BN, int NT, int OP, int ODT>
__device__ __forceinline__ void UnaryTileOp(const GemmParams &p, const uint16_t *stage, int m0, int n0, bool coh)
{
    auto f = [](uint16_t h) {
        const float x = Elem<DT>::Load(h);
        if constexpr (OP == kEwGelu) {
            return GeluTanh(x);
        } else if constexpr (OP == kEwSilu) {
            return Silu(x);
        } else {
            return x;
        }
    };
    if constexpr (ODT == kF32) {
        constexpr int QPR = BN / 4;  // 4-value quarters per row
#pragma unroll 4
        for (int idx = threadIdx.x; idx < BM * QPR; idx += NT) {
            const int row = idx / QPR;
            const int q = idx % QPR;
            const int gm = m0 + row;
            const int gn = n0 + q * 4;
            if (gm >= p.M || gn >= p.N) continue;
            const int slot = (q >> 1) ^ ((row & 31) >> 1);
            const uint2 u = *reinterpret_cast<const uint2 *>(stage + row * BN + slot * 8 + 4 * ((q ^ row) & 1));
            const float o[4] = {f(uint16_t(u.x)), f(uint16_t(u.x >> 16)), f(uint16_t(u.y)), f(uint16_t(u.y >> 16))};
            float *yp = static_cast<float *>(p.uy) + int64_t(gm) * p.ldy + gn;
            if (gn + 4 <= p.N) {
                PutU128(yp, make_uint4(__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]),
                                       __float_as_uint(o[3])), coh);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (gn + e < p.N) PutU32(yp + e, __float_as_uint(o[e]), coh);
            }
        }
    } else {
        constexpr int CPR = BN / 8;
#pragma unroll 4
        for (int idx = threadIdx.x; idx < BM * CPR; idx += NT) {
            const int row = idx / CPR;
            const int ch = idx % CPR;
            const int gm = m0 + row;
            const int gn = n0 + ch * 8;
            if (gm >= p.M || gn >= p.N) continue;
            uint4 u = *reinterpret_cast<const uint4 *>(stage + row * BN + (ch ^ ((row & 31) >> 1)) * 8);
            if (row & 1) u = make_uint4(u.z, u.w, u.x, u.y);
            U16x8 a, r;
            *reinterpret_cast<uint4 *>(a.v) = u;
#pragma unroll
            for (int e = 0; e < 8; ++e) r.v[e] = Elem<ODT>::Store(f(a.v[e]));
            uint16_t *yp = static_cast<uint16_t *>(p.uy) + int64_t(gm) * p.ldy + gn;
            if (gn + 8 <= p.N) {
                PutU128(yp, *reinterpret_cast<const uint4 *>(r.v), coh);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (gn + e < p.N) PutU16(yp + e, r.v[e], coh);
            }
        }
    }
}

// The op and output type are the same for the whole launch: one specialised
// loop each, dispatched once per tile. Tested at run time inside the
// element loop, they turned every element into its own small block behind
// uniform branches, its conversion, exponential and reciprocal chain
// overlapping no other element's (the mm -> GELU epilogue took 190 instead
// of 174 us).
template <int DT, int BM, int BN, int NT>
__device__ __forceinline__ void UnaryTile(const GemmParams &p, const uint16_t *stage, int m0, int n0, bool coh)
{
    auto run = [&](auto op) __attribute__((always_inline)) {
        constexpr int OP = decltype(op)::value;
        if (p.udt == kF32) {
            UnaryTileOp<DT, BM, BN, NT, OP, kF32>(p, stage, m0, n0, coh);
        } else if (p.udt == kBF16) {
            UnaryTileOp<DT, BM, BN, NT, OP, kBF16>(p, stage, m0, n0, coh);
        } else {
            UnaryTileOp<DT, BM, BN, NT, OP, kF16>(p, stage, m0, n0, coh);
        }
    };
    if (p.uop == kEwGelu) {
        run(std::integral_constant<int, kEwGelu>{});
    } else if (p.uop == kEwSilu) {
        run(std::integral_constant<int, kEwSilu>{});
    } else {
        run(std::integral_constant<int, kEwCast>{});
    }
}

// Stage the workgroup's BMxBN tile of C in LDS. acc[i][j][2 sn + sm] is the
// C^T 16x16 sub-block of rows wm*BM/2 + 32i + 16sm.., cols wn*BN/2 + 32j +
// 16sn..: value e of lane l sits at row l%16, col 4*(l/16) + e. Each run of
// 4 columns goes to LDS as one 8-byte write into a row-major tile whose
// 8-byte slots are XOR-swizzled with row & 31 (the rows of one column run hit
// distinct bank pairs). `stage` must hold BM*BN 16-bit values and be free
// (all waves past their last LDS read of the main loop).
template <int DT, int BM, int BN, int MI, int NI>
__device__ __forceinline__ void StageTile(const GemmParams &p, f32x4 (&acc)[MI][NI][4], uint16_t *stage, int n0, int wm,
                                          int wn, int lane)
{
    constexpr int WTN = NI * 32;  // columns per wave
    static_assert(BN >= 128, "slot swizzle needs >= 32 slots per row");
    const int lr = lane & 15;         // row in a 16x16 sub-block
    const int lc = 4 * (lane >> 4);   // first of the lane's four columns in it
#pragma unroll
    for (int j = 0; j < NI; ++j) {
#pragma unroll
        for (int sn = 0; sn < 2; ++sn) {
            const int col = wn * WTN + j * 32 + 16 * sn + lc;
            float b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (p.bias != nullptr) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n0 + col + e < p.N) b[e] = Elem<DT>::Load(p.bias[n0 + col + e]);
            }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int sm = 0; sm < 2; ++sm) {
                    const int row = wm * (BM / 2) + i * 32 + 16 * sm + lr;
                    uint32_t h[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float x = acc[i][j][2 * sn + sm][e];
                        h[e] = p.bias != nullptr ? Elem<DT>::Store(RoundTo<DT>(x) + b[e]) : Elem<DT>::Store(x);
                    }
                    const int slot = (col >> 2) ^ (row & 31);
                    *reinterpret_cast<uint2 *>(stage + row * BN + slot * 4) =
                        make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
                }
        }
    }
}

// The same for a 32x32 accumulator block (lane l: row l % 32, four runs of
// 4 consecutive columns 8 g + 4 (l / 32) ..).
template <int DT, int BM, int BN, int MI, int NI>
__device__ __forceinline__ void StageTile(const GemmParams &p, f32x16 (&acc)[MI][NI], uint16_t *stage, int n0, int wm,
                                          int wn, int lane)
{
    constexpr int WTN = NI * 32;  // columns per wave
    static_assert(BN >= 128, "slot swizzle needs >= 32 slots per row");
    const int lrow = lane & 31;
    const int lhalf = lane >> 5;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int col = wn * WTN + j * 32 + 8 * g + 4 * lhalf;
            float b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (p.bias != nullptr) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n0 + col + e < p.N) b[e] = Elem<DT>::Load(p.bias[n0 + col + e]);
            }
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int row = wm * (BM / 2) + i * 32 + lrow;
                uint32_t h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = acc[i][j][4 * g + e];
                    h[e] = p.bias != nullptr ? Elem<DT>::Store(RoundTo<DT>(x) + b[e]) : Elem<DT>::Store(x);
                }
                const int slot = (col >> 2) ^ (row & 31);
                *reinterpret_cast<uint2 *>(stage + row * BN + slot * 4) =
                    make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
            }
        }
    }
}

// Write the workgroup's BMxBN tile of C: stage it, then every thread copies
// 16-byte row chunks to C (8 lanes cover a 128-byte line), with
// device-scope stores when the launch releases relay tiles.
template <int DT, int BM, int BN, int NT, class ACC>
__device__ __forceinline__ void StoreTile(const GemmParams &p, ACC &acc, uint16_t *stage, int m0, int n0, int wm,
                                          int wn, int lane)
{
    StageTile<DT, BM, BN>(p, acc, stage, n0, wm, wn, lane);
    __syncthreads();
    constexpr int CPR = BN / 8;  // 16-byte chunks per row
    const bool vec = (p.ldc % 8 == 0) && ((reinterpret_cast<uintptr_t>(p.C) & 15) == 0);
    // device-scope stores always: released tiles need them, and written
    // through they also keep the output from evicting the operand tiles the
    // other workgroups of this XCD are still reading from L2
    // (KR_GEMM_STORE=plain|nt for comparison)
    const bool coh = p.store_kind == 0 || p.pub.ctrl != nullptr;
#pragma unroll 4
    for (int idx = threadIdx.x; idx < BM * CPR; idx += NT) {
        const int row = idx / CPR;
        const int ch = idx % CPR;
        const int gm = m0 + row;
        const int gn = n0 + ch * 8;
        if (gm >= p.M || gn >= p.N) continue;
        auto staged = [&](int c) {
            uint4 u = *reinterpret_cast<const uint4 *>(stage + row * BN + (c ^ ((row & 31) >> 1)) * 8);
            return (row & 1) ? make_uint4(u.z, u.w, u.x, u.y) : u;
        };
        uint4 v = staged(ch);
        if (p.rope_cos != nullptr && gn < p.rope_cols) {
            // the partner half of the head is in this tile (tiles start on
            // head boundaries: BN and n0 are multiples of rope_d)
            const int d0 = gn % p.rope_d, half = p.rope_d / 2;
            const uint4 w = staged(d0 < half ? ch + half / 8 : ch - half / 8);
            const int64_t t = int64_t(p.rope_pos0 + gm) * p.rope_d + d0;
            const U16x8 c8 = LoadU16x8(p.rope_cos + t), s8 = LoadU16x8(p.rope_sin + t);
            const uint32_t xv[4] = {v.x, v.y, v.z, v.w}, wv[4] = {w.x, w.y, w.z, w.w};
            uint32_t o[4];
#pragma unroll
            for (int e2 = 0; e2 < 4; ++e2) {
                uint32_t pair = 0;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int e = 2 * e2 + h;
                    const float x = Elem<DT>::Load(uint16_t(xv[e2] >> (16 * h)));
                    const float y = Elem<DT>::Load(uint16_t(wv[e2] >> (16 * h)));
                    const float c = Elem<DT>::Load(c8.v[e]), sn = Elem<DT>::Load(s8.v[e]);
                    const float r = d0 < half ? RopeFirst(x, y, c, sn) : RopeSecond(x, y, c, sn);
                    pair |= uint32_t(Elem<DT>::Store(r)) << (16 * h);
                }
                o[e2] = pair;
            }
            v = make_uint4(o[0], o[1], o[2], o[3]);
        }
        uint16_t *dst = p.C + int64_t(gm) * p.ldc + gn;
        if (vec && gn + 8 <= p.N) {
            if (!coh && p.store_kind == 2) {
                __builtin_nontemporal_store(*reinterpret_cast<const RelayU32x4 *>(&v), reinterpret_cast<RelayU32x4 *>(dst));
            } else {
                PutU128(dst, v, coh);
            }
        } else {
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (gn + e < p.N) PutU16(dst + e, uint16_t(w[e >> 1] >> ((e & 1) * 16)), coh);
        }
    }
    if (p.uy != nullptr) UnaryTile<DT, BM, BN, NT>(p, stage, m0, n0, coh);
}

// SwiGLU epilogue: the in-register relay of the gate/up GEMM to its
// consumer. C's columns hold gate and up interleaved in groups of 8 (cols
// 16q..16q+7 gate, 16q+8..16q+15 up), so a 16x16 C^T sub-block is one group:
// lanes 0-31 hold its gate columns 4 (l / 16) + e, lanes 32-63 the matching
// up columns of the same rows. One v_permlane32_swap per value pairs them
// (lanes 0-31 then hold gate and up of the sub-block's rows 0-15 of sm = 0,
// lanes 32-63 those of sm = 1): act[row, 8q + 4 ((l / 16) & 1) + e] =
// bf16(bf16(silu(bf16(gate))) * bf16(up)), the rounding of the standalone
// SwiGLU kernel reading the stored gate/up tile. C itself is not written.
// The BM x BN/2 act tile is staged in LDS like StoreTile's and leaves as
// full-line 16-byte stores.
template <int DT, int BM, int BN, int MI, int NI>
__device__ __forceinline__ void StageSwiglu(f32x4 (&acc)[MI][NI][4], uint16_t *stage, int wm, int wn, int lane)
{
    constexpr int AW = BN / 2;  // act columns of the tile
    constexpr int WTA = NI * 16;  // act columns per wave
    constexpr int SM = AW / 4 - 1 < 31 ? AW / 4 - 1 : 31;  // the slots of a row the swizzle spans
    const int lr = lane & 15;
    const int hi = lane >> 5;                // after the swap: sub-block rows 16 hi ..
    const int lc = 4 * ((lane >> 4) & 1);    // first act column of the lane in its group
#pragma unroll
    for (int j = 0; j < NI; ++j) {
#pragma unroll
        for (int sn = 0; sn < 2; ++sn) {
            const int acol = wn * WTA + j * 16 + 8 * sn + lc;
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int row = wm * (BM / 2) + i * 32 + 16 * hi + lr;
                uint32_t h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i][j][2 * sn][e]),
                                                                     __float_as_uint(acc[i][j][2 * sn + 1][e]), false,
                                                                     false);
                    const float g = RoundTo<DT>(__uint_as_float(sw[0]));
                    const float u = RoundTo<DT>(__uint_as_float(sw[1]));
                    h[e] = Elem<DT>::Store(RoundTo<DT>(Silu(g)) * u);
                }
                const int slot = (acol >> 2) ^ (row & SM);
                *reinterpret_cast<uint2 *>(stage + row * AW + slot * 4) =
                    make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
            }
        }
    }
}

// The same for 32x32 accumulator blocks: a lane's values v = 0..3 are gate
// columns 8g'+4h+e of group q (g' = 2q) and v = 4..7 the matching up
// columns (g' = 2q + 1), so no lane exchange is needed.
template <int DT, int BM, int BN, int MI, int NI>
__device__ __forceinline__ void StageSwiglu(f32x16 (&acc)[MI][NI], uint16_t *stage, int wm, int wn, int lane)
{
    constexpr int AW = BN / 2;  // act columns of the tile
    constexpr int WTA = NI * 16;  // act columns per wave
    constexpr int SM = AW / 4 - 1 < 31 ? AW / 4 - 1 : 31;  // the slots of a row the swizzle spans
    const int lrow = lane & 31;
    const int lhalf = lane >> 5;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int acol = wn * WTA + j * 16 + q * 8 + 4 * lhalf;
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int row = wm * (BM / 2) + i * 32 + lrow;
                uint32_t h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float g = RoundTo<DT>(acc[i][j][8 * q + e]);
                    const float u = RoundTo<DT>(acc[i][j][8 * q + 4 + e]);
                    h[e] = Elem<DT>::Store(RoundTo<DT>(Silu(g)) * u);
                }
                const int slot = (acol >> 2) ^ (row & SM);
                *reinterpret_cast<uint2 *>(stage + row * AW + slot * 4) =
                    make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
            }
        }
    }
}

template <int DT, int BM, int BN, int NT, class ACC>
__device__ __forceinline__ void StoreTileSwiglu(const GemmParams &p, ACC &acc, uint16_t *stage, int m0, int n0, int wm,
                                                int wn, int lane)
{
    constexpr int AW = BN / 2;  // act columns of the tile
    StageSwiglu<DT, BM, BN>(acc, stage, wm, wn, lane);
    __syncthreads();
    constexpr int CPR = AW / 8;
    constexpr int SM = AW / 4 - 1 < 31 ? AW / 4 - 1 : 31;
    const int64_t a0 = n0 / 2;
    const int acols = p.N / 2;
#pragma unroll 4
    for (int idx = threadIdx.x; idx < BM * CPR; idx += NT) {
        const int row = idx / CPR;
        const int ch = idx % CPR;
        const int gm = m0 + row;
        const int gn = int(a0) + ch * 8;
        if (gm >= p.M || gn >= acols) continue;
        uint4 v = *reinterpret_cast<const uint4 *>(stage + row * AW + (ch ^ ((row & SM) >> 1)) * 8);
        if (row & 1) v = make_uint4(v.z, v.w, v.x, v.y);
        PutU128(p.epi_act + int64_t(gm) * p.ld_act + gn, v, p.store_kind == 0 || p.pub.ctrl != nullptr);
    }
}

template <int DT, int BM, int BN>
__global__ void __attribute__((amdgpu_flat_work_group_size(kThreads, kThreads),
                               amdgpu_waves_per_eu(BM * BN >= 256 * 128 ? 1 : 2, BM * BN >= 256 * 128 ? 1 : 2)))
GemmKernel(GemmParams p)
{
    constexpr int MI = BM / 64;   // 32-row blocks per wave
    constexpr int NI = BN / 64;   // 32-col blocks per wave
    constexpr int AL = BM * kRowChunks / kThreads;  // A chunks per thread per stage
    constexpr int BL = BN * kRowChunks / kThreads;
    constexpr int STAGE = (BM + BN) * kBK;           // elements per LDS stage

    __shared__ __attribute__((aligned(16))) uint16_t smem[2 * STAGE];

    if (int(blockIdx.x) >= p.gemm_wgs) {
        TailSwiglu<DT>(p);
        return;
    }
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave >> 1;
    const int wn = wave & 1;

    int tm, tn;
    TileOf(blockIdx.x, p.tiles_m, p.tiles_n, BM, p.order_rows, p.group_m, tm, tn);
    const int m0 = tm * BM;
    const int n0 = tn * BN;
    RelayWaitRows(p.wait, m0, min(m0 + BM, p.M));

    const int lrow = tid >> 3;       // 0..31
    const int lchunk = tid & 7;

    uint4 ra[AL], rb[BL];

    auto load_global = [&](int kt) {
        const int kc = kt * kBK + lchunk * 8;
        const bool kin = kc < p.K;
#pragma unroll
        for (int j = 0; j < AL; ++j) {
            const int r = lrow + 32 * j;
            const int gm = m0 + r;
            if (kin && gm < p.M) {
                ra[j] = *reinterpret_cast<const uint4 *>(p.A + int64_t(gm) * p.lda + kc);
            } else {
                ra[j] = make_uint4(0, 0, 0, 0);
            }
        }
#pragma unroll
        for (int j = 0; j < BL; ++j) {
            const int r = lrow + 32 * j;
            const int gn = n0 + r;
            if (kin && gn < p.N) {
                rb[j] = *reinterpret_cast<const uint4 *>(p.Bt + int64_t(gn) * p.ldb + kc);
            } else {
                rb[j] = make_uint4(0, 0, 0, 0);
            }
        }
    };

    auto store_lds = [&](int stage) {
        uint16_t *As = smem + stage * STAGE;
        uint16_t *Bs = As + BM * kBK;
#pragma unroll
        for (int j = 0; j < AL; ++j) {
            const int r = lrow + 32 * j;
            *reinterpret_cast<uint4 *>(As + r * kBK + Swz(r, lchunk) * 8) = ra[j];
        }
#pragma unroll
        for (int j = 0; j < BL; ++j) {
            const int r = lrow + 32 * j;
            *reinterpret_cast<uint4 *>(Bs + r * kBK + Swz(r, lchunk) * 8) = rb[j];
        }
    };

    f32x4 acc[MI][NI][4];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[i][j][q][v] = 0.0f;

    const int nk = (p.K + kBK - 1) / kBK;
    load_global(0);
    store_lds(0);
    __syncthreads();

    const int frow = lane & 15;
    const int fq = lane >> 4;

    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
        if (kt + 1 < nk) load_global(kt + 1);
        const uint16_t *As = smem + cur * STAGE;
        const uint16_t *Bs = As + BM * kBK;
        // two k32 steps: lane l reads row l % 16 of each 16-row fragment,
        // 16-byte chunk 4 ks + l / 16
#pragma unroll
        for (int ks = 0; ks < kBK / 32; ++ks) {
            const int chunk = ks * 4 + fq;
            uint4 fa[MI][2], fb[NI][2];
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int sm = 0; sm < 2; ++sm) {
                    const int r = wm * (BM / 2) + i * 32 + 16 * sm + frow;
                    fa[i][sm] = *reinterpret_cast<const uint4 *>(As + r * kBK + Swz(r, chunk) * 8);
                }
#pragma unroll
            for (int j = 0; j < NI; ++j)
#pragma unroll
                for (int sn = 0; sn < 2; ++sn) {
                    const int r = wn * (BN / 2) + j * 32 + 16 * sn + frow;
                    fb[j][sn] = *reinterpret_cast<const uint4 *>(Bs + r * kBK + Swz(r, chunk) * 8);
                }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        acc[i][j][q] = Mfma<DT>(fb[j][q >> 1], fa[i][q & 1], acc[i][j][q]);
        }
        if (kt + 1 < nk) store_lds(cur ^ 1);
        __syncthreads();
    }

    // (SwigluTile: no launch asks 128-column tiles of this kernel for SwiGLU)
    if constexpr (BN >= 256) {
        if (p.epi_act != nullptr) {
            StoreTileSwiglu<DT, BM, BN, kThreads>(p, acc, smem, m0, n0, wm, wn, lane);
        } else {
            StoreTile<DT, BM, BN, kThreads>(p, acc, smem, m0, n0, wm, wn, lane);
        }
    } else {
        StoreTile<DT, BM, BN, kThreads>(p, acc, smem, m0, n0, wm, wn, lane);
    }
    if (p.pub.ctrl != nullptr) {
        const int tile = m0 / p.pub.rows_per_tile;
        int *slot = reinterpret_cast<int *>(smem);  // the tile stage is free
        const int a = RelayArriveIndexed(p.pub, tile, slot);
        if (p.rn_y != nullptr)
            NormTail<DT, kThreads / 64, BM * BN >= 256 * 128 ? 1 : 2>(p, tile, p.pub.arrivals, a, slot + 1);
    }
    RelayFinish(p.wait);
}

// Stream-K partial sums move as 16-byte device-scope accesses (written
// through to memory / read past this XCD's L2, which may hold stale lines of
// the workspace from an earlier launch).
__device__ __forceinline__ void PutF32x4Dev(float *p, float a, float b, float c, float d)
{
    const RelayU32x4 w = {__float_as_uint(a), __float_as_uint(b), __float_as_uint(c), __float_as_uint(d)};
    // two wait states before the data VGPRs may be rewritten (as PutU128)
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(w) : "memory");
}

// Eight 16-byte device-scope loads p + u * stride (floats), in flight
// together; returns once all have landed.
__device__ __forceinline__ void GetF32x4x8Dev(const float *p, int64_t stride, RelayU32x4 (&r)[8])
{
    asm volatile(
        "global_load_dwordx4 %0, %8, off sc1\n\t"
        "global_load_dwordx4 %1, %9, off sc1\n\t"
        "global_load_dwordx4 %2, %10, off sc1\n\t"
        "global_load_dwordx4 %3, %11, off sc1\n\t"
        "global_load_dwordx4 %4, %12, off sc1\n\t"
        "global_load_dwordx4 %5, %13, off sc1\n\t"
        "global_load_dwordx4 %6, %14, off sc1\n\t"
        "global_load_dwordx4 %7, %15, off sc1\n\t"
        "s_waitcnt vmcnt(0)"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
        : "v"(p), "v"(p + stride), "v"(p + 2 * stride), "v"(p + 3 * stride), "v"(p + 4 * stride),
          "v"(p + 5 * stride), "v"(p + 6 * stride), "v"(p + 7 * stride)
        : "memory");
}

// ---------------------------------------------------------------------------
#include "kr_gemm_pipe.inc"

// KR_GEMM_SIMPLE=1 routes every shape through GemmKernel (A/B comparison of
// the two main loops; both give identical bits).
bool ForceSimple()
{
    static const bool v = [] {
        const char *e = std::getenv("KR_GEMM_SIMPLE");
        return e != nullptr && *e == '1';
    }();
    return v;
}

int StoreKind()
{
    static const int v = [] {
        const char *e = std::getenv("KR_GEMM_STORE");
        if (e == nullptr) return 0;
        return std::string(e) == "plain" ? 1 : std::string(e) == "nt" ? 2 : 0;
    }();
    return v;
}

// Row blocks per raster group of a launch without relay order
// (KR_GEMM_GROUP_M, default 4; 0 = all rows, a column at a time); it changes
// timing only, never the bits.
int RasterGroupM()
{
    static const int v = [] {
        const char *e = std::getenv("KR_GEMM_GROUP_M");
        return e != nullptr ? std::max(0, std::atoi(e)) : 4;
    }();
    return v;
}

// Waves per workgroup of the 256x256 pipelined kernel (KR_GEMM_WAVES: 8
// default, two per SIMD; 4 = one per SIMD); it changes timing only, never
// the bits. Measured on MI355X (cold operands): 4096^3 138 -> 130 us, the
// 2048x4608x3584 QKV 112 -> 104 us, lm_head 2068 -> 2036 us.
int PipeWaves()
{
    static const int v = [] {
        const char *e = std::getenv("KR_GEMM_WAVES");
        return e != nullptr && std::atoi(e) == 4 ? 4 : 8;
    }();
    return v;
}

// Main loop of the 8-wave 256x256 kernel (KR_GEMM_LOOP): 2 (default) =
// register-staged refills spread evenly over each stage, 0 = two 64-deep
// direct-to-LDS stages refilled in a burst after each stage's barrier.
// Timing only, never the bits. Measured on MI355X (us, 0 / 2): 4096^3
// 126.7 / 118.5, gate/up 2048x37888x3584 561 / 529, QKV 2048x4608x3584
// 103 / 85, lm_head 2048x152064x3584 1967 / 1871. Two other schedules
// measured slower than both: the two waves of a SIMD alternating memory and
// MFMA phases on a direct-to-LDS ring (4096^3 140 us), and a ring of four or
// five 32-deep direct-to-LDS stages (142 us: half-line requests). The same
// alternation on the staged refill (per k32 step: fragment reads and half a
// stage of refill, then 32 MFMAs, a barrier after each phase) gave the same
// bits in the same time (4096^3 111.0 against 110.1 us). The 4-wave 256x128 and
// 128x256 kernels keep their three-stage direct-to-LDS ring, which already
// spreads its refills: staged, they measured 4-8% slower.
int MainLoopMode()
{
    static const int v = [] {
        const char *e = std::getenv("KR_GEMM_LOOP");
        return e != nullptr && std::atoi(e) == 0 ? 0 : 2;
    }();
    return v;
}

// L2 prefetch distance of the pipelined kernel in K stages (KR_GEMM_PF: 0
// default = off, 2, 4); it changes timing only, never the bits.
int PrefetchStages()
{
    static const int v = [] {
        const char *e = std::getenv("KR_GEMM_PF");
        return e != nullptr ? std::atoi(e) : 0;
    }();
    return v;
}

// Stream-K plan of a launch: G resident workgroups over tiles x nk
// iterations, at most pmax pieces per tile.
struct StreamKPlan {
    int G = 0, tiles = 0, nk = 0, pmax = 0;
    int bm = 256, bn = 256;  // below 256 rows: GemmSplitKernel, every tile in G / tiles pieces
    size_t WsBytes() const { return size_t(tiles) * pmax * bm * bn * 4; }
};

int CuCount()
{
    static const int v = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 256;
        return n > 0 ? n : 256;
    }();
    return v;
}

// Whether a launch of bm x 128 tiles takes the deep ring: at most one
// workgroup per CU, and for 128 rows a K of more than six stages. There its
// four stages are filled at once and bring nothing to a K that ends with them,
// while the kernel is slower to start (2048x1280, 160 tiles, two-stage ring
// against deep: K 128 5.6 / 6.2 us, K 384 7.4 / 7.7, K 512 9.5 / 8.5;
// 2048x2048, 256 tiles: K 192 6.3 / 6.9, K 384 8.7 / 8.2). 64 row tiles
// are faster with it from K 64 on (1024x1024x128 5.6 -> 4.7).
bool DeepGrid(int bm, int bn, int M, int N, int K)
{
    if (bm * bn >= 256 * 128 || bn != 128 || (bm == 128 && K <= 6 * kPipeK)) return false;
    return int64_t((M + bm - 1) / bm) * ((N + bn - 1) / bn) <= CuCount();
}

// The larger of two row strides (elements); one that steps backwards counts
// as the largest.
int64_t RowSpan(int64_t lda, int64_t ldb) { return lda < 0 || ldb < 0 ? INT64_MAX : std::max(lda, ldb); }

// Whether the launch's 256-wide tiles run the wide loop: K of at least 32
// stages (its 4-wave prologue and epilogue, one wave per SIMD, cost more than
// the 8-wave kernel's: 16384x2048x1024 71 -> 74 us), and workgroups for three
// quarters of the CUs in 256x128 and 128x256 tiles (1024x3584x3584, 112 tiles,
// 48.6 against 49.6 us; 1536x4096x4096, 192 tiles, 52.5 -> 51.1;
// 2048x4096x12288, 256 tiles, 176 -> 167).
// For 256x256 tiles, whose two-stage ring asks for a stage's data no earlier
// than the stage before it, only where the 8-wave loop measured slower:
// * four fifths of the CUs (8-wave / wide, us: 192 tiles 2048x6144x4096 85.5 /
//   89, 16384x520x2048 45 / 47; 208 tiles 4096x3328x4096 90 / 87; 256
//   tiles 4096x4096x8192 204 / 190);
// * operands that come from the 256 MB Infinity Cache rather than HBM: all of
//   them together (4096x3584: K 16384, 252 MB, 383 / 370; K 18944, 291 MB, 434 /
//   467; 4096^2x16384, 268 MB, 409 / 460; 16384x1024: K 6144, 214 MB, 156 /
//   149; K 8192, 285 MB, 212 / 220), or, over more than one round of
//   workgroups, A in half of it (8192x8192: K 8192, A 134 MB, 801 / 754; K
//   14336, A 235 MB, 1422 / 1451; 8192x4096x12288, A 201 MB, 602 / 617;
//   4096x12288: K 16384, A 134 MB, 1211 / 1194; K 18944, A 155 MB, 1383 / 1412);
// * no Add+RMSNorm consumer: its rows take 8 waves per workgroup faster
//   (4096x3584x3584 108 / 113, 4096x4096x12288 316 / 324).
// Its tile rows are addressed by unsigned 32-bit byte offsets: `stride`
// (RowSpan) must keep 256 of them below 4 GB.
bool WideLoop(int bm, int bn, int M, int N, int K, int64_t stride, bool norm)
{
    if (stride >= (int64_t(1) << 23)) return false;
    if (K % kPipeK != 0 || K < 32 * kPipeK || ForceSimple() || MainLoopMode() != 2 || PipeWaves() != 8 ||
        PrefetchStages() != 0)
        return false;
    const int64_t tiles = int64_t((M + bm - 1) / bm) * ((N + bn - 1) / bn), cus = CuCount();
    if (bm * bn == 256 * 128) return tiles * 4 >= cus * 3;
    if (bm != 256 || bn != 256 || norm || tiles * 5 < cus * 4) return false;
    constexpr int64_t kCache = int64_t(256) << 20;  // bytes
    return 2 * int64_t(K) * (int64_t(M) + N) < kCache || (tiles > cus && 4 * int64_t(K) * M <= kCache);
}

// The loop a launch of bm x bn tiles runs over K: the simple kernel where
// K % 64 != 0 or KR_GEMM_SIMPLE=1; the 8-wave kernel for 192x256 and 256x256
// (stream-K or data-parallel) unless KR_GEMM_WAVES=4; the wide loop for
// 256-wide tiles with K long enough; the deep ring for a small tile whose
// grid has at most one workgroup per CU; the 4-wave ring for the others.
GemmLoop LoopOf(int bm, int bn, int M, int N, int K, int64_t stride, bool sk, bool norm)
{
    if (bm == 192) return GemmLoop::kStaged;
    if (K % kPipeK != 0 || ForceSimple()) return GemmLoop::kSimple;
    if (!sk && WideLoop(bm, bn, M, N, K, stride, norm)) return GemmLoop::kWide;
    if (bm == 256 && bn == 256 && (sk || PipeWaves() == 8)) return GemmLoop::kStaged;
    if (DeepGrid(bm, bn, M, N, K)) return GemmLoop::kDeep;
    return GemmLoop::kRing;
}

// The tile of a SwiGLU epilogue launch in place of t. The simple kernel and
// the two-stage ring of the small tiles have no SwiGLU on 128 columns: its code
// beside the plain epilogue cost every plain launch of them 0.1 to 0.4 us
// (2048x1280x128 5.65 -> 5.80, 640x128x1000 17.4 -> 17.8). Such a launch takes
// 256 columns.
GemmTile SwigluTile(GemmTile t, GemmLoop loop)
{
    if (t.bn >= 256 || (loop != GemmLoop::kSimple && (t.bm * t.bn >= 256 * 128 || loop == GemmLoop::kDeep))) return t;
    return {t.bm >= 256 ? 256 : 128, 256};
}

using GemmFn = void (*)(GemmParams);

// The kernel of LoopOf's choice, and its block size.
template <int DT, int BM, int BN>
GemmFn PickGemmKernel(int M, int N, int K, int64_t stride, bool sk, bool norm, int &threads)
{
    [[maybe_unused]] const GemmLoop loop = LoopOf(BM, BN, M, N, K, stride, sk, norm);
    if constexpr (BM == 192) {
        // 192x256: the 8-wave staged kernel only (GemmLaunch picks this tile
        // only where that kernel runs)
        static_assert(BN == 256, "192-row tiles pair with 256 columns");
        if (sk || K % kPipeK != 0 || ForceSimple() || MainLoopMode() != 2)
            throw std::logic_error("gemm: 192x256 tiles run the staged kernel only");
        threads = 512;
        return GemmPipeKernel<DT, BM, BN, 0, 8, false, 2>;
    } else {
        if constexpr (BM * BN >= 128 * 256) {
            if (loop == GemmLoop::kWide) {
                threads = kThreads;
                return GemmPipeKernel<DT, BM, BN, 0, 4, false, 3>;
            }
        }
        if constexpr (BM == 256 && BN == 256) {
            if (loop == GemmLoop::kStaged) {
                threads = 512;
                if (sk)
                    return MainLoopMode() == 2 ? GemmPipeKernel<DT, BM, BN, 0, 8, true, 2>
                                               : GemmPipeKernel<DT, BM, BN, 0, 8, true>;
                return MainLoopMode() == 2 ? GemmPipeKernel<DT, BM, BN, 0, 8, false, 2>
                                           : GemmPipeKernel<DT, BM, BN, 0, 8>;
            }
        }
        threads = kThreads;
        if (loop == GemmLoop::kSimple) return GemmKernel<DT, BM, BN>;
        if constexpr (BM * BN < 256 * 128 && BN == 128) {
            if (loop == GemmLoop::kDeep) return GemmPipeKernel<DT, BM, BN, 0, 4, false, 0, DeepStages<BM, BN>()>;
        }
        switch (PrefetchStages()) {
        case 2: return GemmPipeKernel<DT, BM, BN, 2, 4>;
        case 4: return GemmPipeKernel<DT, BM, BN, 4, 4>;
        default: return GemmPipeKernel<DT, BM, BN, 0, 4>;
        }
    }
}

// Workgroups of that kernel one CU holds at once, from the runtime's
// occupancy query on the exact instantiation (registers, LDS, waves);
// cached per (dtype, tile, stream-K, loop).
template <int DT, int BM, int BN>
int GemmWgsPerCu(int M, int N, int K, int64_t stride, bool sk, bool norm)
{
    static int cache[2][5] = {};  // 0: not asked yet
    int &c = cache[sk][int(LoopOf(BM, BN, M, N, K, stride, sk, norm))];
    if (c == 0) {
        int threads = 0;
        const GemmFn fn = PickGemmKernel<DT, BM, BN>(M, N, K, stride, sk, norm, threads);
        int n = 0;
        Check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(fn), threads, 0),
              "gemm occupancy");
        if (n < 1) throw std::runtime_error("gemm: kernel does not fit a CU");
        c = n;
    }
    return c;
}

int GemmWgsPerCu(int dt, int bm, int bn, int M, int N, int K, int64_t stride, bool sk, bool norm)
{
    const bool bf = dt == kBF16;
#define KR_OCC_CASE(BM_, BN_) \
    if (bm == BM_ && bn == BN_) return bf ? GemmWgsPerCu<kBF16, BM_, BN_>(M, N, K, stride, sk, norm) \
                                                  : GemmWgsPerCu<kF16, BM_, BN_>(M, N, K, stride, sk, norm);
    KR_OCC_CASE(256, 256)
    KR_OCC_CASE(192, 256)
    KR_OCC_CASE(256, 128)
    KR_OCC_CASE(128, 256)
    KR_OCC_CASE(128, 128)
    KR_OCC_CASE(64, 128)
    KR_OCC_CASE(64, 256)
#undef KR_OCC_CASE
    throw std::runtime_error("gemm: unsupported tile " + std::to_string(bm) + "x" + std::to_string(bn));
}

// The Add+RMSNorm relay consumer waits inside the producer's workgroups for
// the other producer workgroups of its relay tile, and is worth it where
// those fit the device at once: workgroups are dispatched in id order (per
// XCD) and a relay tile's are consecutive ids, so every earlier tile's are
// resident or finished then; a split grid must fit as a whole. (Where the
// device is not free for them the waits end by patience, NormTail.) The
// device's slots come from the occupancy of the kernel the launch runs.
bool NormRelayResident(int dt, int bm, int bn, int M, int N, int K, int rows_per_tile, int sk_wgs)
{
    if (sk_wgs > 0 && bm < 256) return sk_wgs <= CuCount();  // GemmSplitKernel: one per CU
    if (sk_wgs > 0) return sk_wgs <= CuCount() * GemmWgsPerCu(dt, 256, 256, M, N, K, K, true, true);
    if (rows_per_tile <= 0 || rows_per_tile % bm != 0 || M % rows_per_tile != 0) return false;
    const int per = (rows_per_tile / bm) * ((N + bn - 1) / bn);
    return per <= CuCount() * GemmWgsPerCu(dt, bm, bn, M, N, K, K, false, true);
}

// Estimated time (us) of a 256x256 split in S pieces (the last one sums all
// partials alone, so the fix-up grows with S).
double Split256Us(int K, int S)
{
    return 21.0 + (K / kPipeK + S - 1) / S * 1.5 + 2.0 * S;
}

// Estimated time (us) of a product in bm x 128 tiles, one workgroup per CU on
// the deep ring, each tile in S pieces of K (two stages or more in each);
// negative when that does not fit.
// Fitted to M 37..1500 at the projections of the three shipped models (within
// 15%): a launch costs 6, a stage 0.24 (64 rows) / 0.32 (128) alone and 0.38 /
// 0.59 with every CU loading, a fix-up 2 plus 0.5 / 1.4 a piece.
double SmallTileUs(int bm, int S, int M, int N, int K)
{
    const int tiles = ((M + bm - 1) / bm) * ((N + 127) / 128), G = tiles * S, nk = K / kPipeK;
    if (K % kPipeK != 0 || G > CuCount() || (S > 1 && nk < 2 * S)) return -1.0;
    const double load = double(G) / CuCount();
    const double stage = bm == 64 ? 0.24 + 0.14 * load : 0.32 + 0.27 * load;
    const double fix = S > 1 ? 2.0 + (bm == 64 ? 0.5 : 1.4) * S : 0.0;
    return 6.0 + (nk + S - 1) / S * stage + fix;
}

// Split plan of a small product (GemmSplitKernel): the cheapest of 64 and 128
// row tiles in up to 16 pieces, taken when it beats the same tiles unsplit and
// the 256x256 split `big` (its pieces; 0: none). Below 1920 rows only: from
// there the plan, the workspace it reports and the bits are those of the
// 256x256 split, which callers have been told. The line is not where the small
// plan stops paying (us, 256x256 split / small plan / whole tiles: 2048x896x4864
// 46.5 / 25.8 / 25.6, 2560x896x4864 47.8 / 31.9 / 31.8, 2048x1024x4096 43.2 /
// 24.7 / 23.5, 2048x512x4096 41.8 / 19.1 / 21.6; 1919 rows of each take 24.8,
// 23.4 and 17.3).
bool PlanSplit(int M, int N, int K, int big, StreamKPlan &pl)
{
    if (M >= 1920 || K % kPipeK != 0) return false;
    double best = big > 1 ? Split256Us(K, big) : 1e30;
    int bm = 0, S = 0;
    for (int b : {64, 128}) {
        for (int s = 1; s <= 16; ++s) {
            const double us = SmallTileUs(b, s, M, N, K);
            if (us < 0.0 || us >= best) continue;
            best = us;
            bm = b;
            S = s;
        }
    }
    if (bm == 0) return false;
    pl.bm = bm;
    pl.bn = 128;
    pl.nk = K / kPipeK;
    pl.tiles = ((M + bm - 1) / bm) * ((N + 127) / 128);
    pl.pmax = S;
    pl.G = S * pl.tiles;
    return true;
}

// Tile of a launch that releases relay tiles or shares its CUs, or that the
// estimates below do not cover.
GemmTile PickRelayTile(int M, int N, int relay_rows, bool coresident)
{
    // Candidates from most to least data reuse; take the first that keeps the
    // device busy (>= 2 full waves of workgroups, or whole waves) or, failing
    // that, the one with the best wave efficiency. A GEMM whose 128x128 tiles
    // give every workgroup a CU of its own takes them: with so few workgroups
    // each CU's load path is the limit, and smaller tiles put more CUs to
    // work.
    static const GemmTile cands[] = {{256, 256}, {256, 128}, {128, 256}, {128, 128}, {64, 256}};
    const int cus = 256;
    if ((relay_rows == 0 || relay_rows % 128 == 0) && ((M + 127) / 128) * ((N + 127) / 128) <= cus)
        return {128, 128};
    GemmTile best{-1, -1};
    double best_eff = -1.0;
    for (const GemmTile &t : cands) {
        if (relay_rows > 0 && relay_rows % t.bm != 0) continue;
        if (coresident && t.bm * t.bn >= 256 * 256) continue;
        const int tiles = ((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
        const int slots = cus * (t.bm * t.bn >= 256 * 128 ? 1 : 2);
        // enough workgroups for two rounds, or whole rounds exactly
        if (tiles >= 2 * slots || tiles % slots == 0) return t;
        const double work = double(t.bm) * t.bn;  // per-workgroup work unit
        const double eff = double(tiles) * work / (double((tiles + slots - 1) / slots) * slots * work);
        const double score = eff * (t.bm * t.bn >= 256 * 128 ? 1.0 : 0.85);
        if (score > best_eff) {
            best_eff = score;
            best = t;
        }
    }
    return best;
}

// Pieces of the 256x256 split (below).
int Split256Pieces(int M, int N, int tiles, int nk)
{
    const GemmTile dp = PickRelayTile(M, N, 0, false);
    const int dp_tiles = ((M + dp.bm - 1) / dp.bm) * ((N + dp.bn - 1) / dp.bn);
    const int dp_slots = CuCount() * (dp.bm * dp.bn >= 256 * 128 ? 1 : 2);
    const int dp_rounds = (dp_tiles + dp_slots - 1) / dp_slots;
    const double fill = double(dp_tiles) / (double(dp_rounds) * dp_slots);
    static const bool longk = [] {
        const char *e = std::getenv("KR_GEMM_SK_LONGK");
        return e == nullptr || std::atoi(e) != 0;
    }();
    static const int longk_nk = [] {
        const char *e = std::getenv("KR_GEMM_SK_LONGK_NK");
        return e != nullptr ? std::max(32, std::atoi(e)) : 256;
    }();
    if (fill >= 0.6 && !(longk && fill < 0.9 && nk >= longk_nk)) return 0;
    const int S = std::min(CuCount() / tiles, nk / 16);
    // 128x128 tiles run one workgroup per CU on the deep ring: where they
    // fill 60% of the CUs they stay whole unless the split is estimated
    // faster (4096x1024x4096: 38 us against 57 in four pieces; 1024x3584x18944:
    // 160 against 137)
    if (dp.bm == 128 && dp.bn == 128 && dp_tiles >= 0.6 * CuCount() && dp_tiles <= CuCount() &&
        SmallTileUs(128, 1, M, N, nk * kPipeK) < Split256Us(nk * kPipeK, std::max(S, 1)))
        return 0;
    return S;
}

// Stream-K plan of a GEMM whose data-parallel tiling leaves CUs idle.
// Small products first: see PlanSplit. Otherwise:
// Default: an exact split of K over 256x256 tiles, S = CUs / tiles pieces per
// tile, each piece at least 16 K stages (S >= 2), so every workgroup runs one
// piece and the workgroups of an XCD walk K in step on a compact patch of
// tiles; where the best data-parallel tiling fills less than 60% of the
// device's workgroup slots, or less than 90% with K of at least 256 stages
// (16384), where two long pieces per 256x256 tile amortise the fix-up. The
// last piece to finish sums all S partials alone, so short pieces lose to
// that fix-up: 2048x896x4864 in 2 pieces 65.7 us, 4 pieces (19 stages) 53.6 (46.5
// on the present loop), 8 pieces (9.5 stages) 78.2; 2048x896x896 with 2 pieces
// of 7 stages 32.3 against 21.0. Both rules were fitted to the two-stage ring
// and the staged loop: the whole tiles took 67.1 us for 2048x896x4864 (25.6 on the
// deep ring now) and 248 for 2048x3584x18944 in the 7B prefill, against 226 in
// two pieces of 148 stages. On the wide loop the whole 256x128 tiles take 225
// us against the split's 231 alone and 257 against 260 in the prefill of one
// card (KR_GEMM_SK_LONGK=0): the long-K split no longer gains there. Spreading the iterations of every tile over all 256 CUs
// instead (pieces of uneven length at different K offsets, sharing no
// operand lines) took 369 us for 2048x3584x18944. KR_GEMM_SK_WGS=G forces that
// even spread over G workgroups (a measurement aid).
bool PlanStreamK(int M, int N, int K, StreamKPlan &pl)
{
    pl = StreamKPlan{};
    if (K % kPipeK != 0) return false;
    pl.tiles = ((M + 255) / 256) * ((N + 255) / 256);
    pl.nk = K / kPipeK;
    if (const char *e = std::getenv("KR_GEMM_SK_WGS")) {
        if (M < 256 || N < 256) return false;
        pl.G = std::max(1, std::atoi(e));
        if (pl.tiles >= pl.G || int64_t(pl.tiles) * pl.nk < 4 * int64_t(pl.G)) return false;
    } else {
        const int S = M < 256 || N < 256 ? 0 : Split256Pieces(M, N, pl.tiles, pl.nk);
        StreamKPlan small;
        if (PlanSplit(M, N, K, S, small)) {
            if (small.pmax < 2) return false;  // best as one piece per tile: data-parallel
            pl = small;
            return true;
        }
        if (S < 2) return false;
        pl.G = S * pl.tiles;
    }
    const int64_t I = int64_t(pl.tiles) * pl.nk;
    if ((I + pl.G - 1) / pl.G > pl.nk) return false;  // a run spans at most two pieces
    auto owner = [&](int64_t x) { return int(((x + 1) * pl.G - 1) / I); };
    pl.pmax = 1;
    for (int t = 0; t < pl.tiles; ++t)
        pl.pmax = std::max(pl.pmax, owner(int64_t(t) * pl.nk + pl.nk - 1) - owner(int64_t(t) * pl.nk) + 1);
    return true;
}

// With the Add+RMSNorm consumer a workgroup finishes one tile at most (not so in
// the even spread of KR_GEMM_SK_WGS).
bool SplitNormOk(const StreamKPlan &pl) { return pl.G <= CuCount() && pl.G == pl.tiles * pl.pmax; }

// A split launch can release any relay tiles of whole 64-row blocks: a
// finisher arrives on every relay tile its rows touch (ArriveRows), whether
// they are whole row blocks or not.
bool SplitPubOk(int M, int R) { return R > 0 && R % 64 == 0 && M % R == 0; }

template <int DT, int BM, int BN>
void LaunchSplit(const GemmParams &base, const StreamKPlan &pl, hipStream_t stream)
{
    GemmParams p = base;
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN - 1) / BN;
    if (p.tiles_m * p.tiles_n != pl.tiles || pl.G != pl.tiles * pl.pmax || pl.G > CuCount())
        throw std::logic_error("gemm: split plan mismatch");
    p.order_rows = 0;
    p.group_m = RasterGroupM();
    p.sk_wgs = pl.G;
    p.sk_pmax = pl.pmax;
    p.gemm_wgs = pl.G;
    hipLaunchKernelGGL((GemmSplitKernel<DT, BM, BN, DeepStages<BM, BN>()>), dim3(pl.G), dim3(kThreads), 0, stream, p);
    Check(hipGetLastError(), "gemm split launch");
}

template <int DT, int BM, int BN>
void LaunchTyped(const GemmParams &base, int order_rows, int tail_tiles, hipStream_t stream,
                 const StreamKPlan *sk = nullptr)
{
    GemmParams p = base;
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN - 1) / BN;
    // relay order needs whole relay tiles of whole row blocks
    auto whole = [&](int rows) { return rows > 0 && rows % BM == 0 && p.tiles_m % (rows / BM) == 0; };
    p.order_rows = 0;
    if (p.pub.ctrl != nullptr && sk != nullptr) {
        // stream-K: each tile's finisher arrives on every relay tile its rows
        // touch (ArriveRows counts the arrivals)
        if (!SplitPubOk(p.M, p.pub.rows_per_tile))
            throw std::runtime_error("gemm: stream-K relay tiles must be whole 64-row blocks dividing M");
    } else if (p.pub.ctrl != nullptr) {
        if (!whole(p.pub.rows_per_tile)) throw std::runtime_error("relay tile rows must be a multiple of BM dividing M");
        p.pub.arrivals = (p.pub.rows_per_tile / BM) * p.tiles_n;
        p.order_rows = p.pub.rows_per_tile;
        if (order_rows > 0) {
            if (order_rows % p.pub.rows_per_tile != 0 || !whole(order_rows))
                throw std::runtime_error("gemm: order_rows must be a multiple of the relay tile dividing M");
            p.order_rows = order_rows;
        }
    } else if (p.wait.ctrl != nullptr && p.wait.row_off == 0 && whole(p.wait.prod_rows)) {
        p.order_rows = p.wait.prod_rows;  // the rows that are released first run first
    }
    p.gemm_wgs = p.tiles_m * p.tiles_n;
    p.group_m = RasterGroupM();
    if (p.rn_y != nullptr) {
        if (sk == nullptr && p.order_rows != p.pub.rows_per_tile)
            throw std::runtime_error("gemm: the Add+RMSNorm relay consumer needs the default relay-tile order");
        if (!NormRelayResident(DT, BM, BN, p.M, p.N, p.K, p.pub.rows_per_tile, sk != nullptr ? sk->G : 0))
            throw std::runtime_error("gemm: a relay tile's producer workgroups do not fit the device at once; "
                                     "the Add+RMSNorm relay consumer would wait on workgroups not yet placed");
        // a grid resident as a whole releases every tile at about the same
        // time whatever the order: keep the grouped raster (square patches
        // per XCD, less operand traffic than relay-tile order)
        if (sk == nullptr && p.gemm_wgs <= CuCount() * GemmWgsPerCu<DT, BM, BN>(p.M, p.N, p.K, RowSpan(p.lda, p.ldb), false, true))
            p.order_rows = 0;
    }
    if (sk != nullptr) {
        if (BM != 256 || BN != 256 || sk->tiles != p.gemm_wgs) throw std::logic_error("gemm: stream-K plan mismatch");
        p.sk_wgs = sk->G;
        p.sk_pmax = sk->pmax;
        p.gemm_wgs = sk->G;
    }
    int grid_x = p.gemm_wgs;
    if (p.tail_act != nullptr) {
        p.tail_wpt = 256;  // one per CU of the device: enough to fill the idle CUs of the last round
        grid_x += tail_tiles * p.tail_wpt;
    }
    const dim3 grid(grid_x);
    int threads = 0;
    const GemmFn fn = PickGemmKernel<DT, BM, BN>(p.M, p.N, p.K, RowSpan(p.lda, p.ldb), sk != nullptr, p.rn_y != nullptr, threads);
    void *args[] = {&p};
    Check(hipLaunchKernel(reinterpret_cast<const void *>(fn), grid, dim3(threads), args, 0, stream), "gemm launch");
}

}  // namespace

namespace {

// Cheaper of 128 and 64 row tiles, one workgroup per CU on the deep ring
// (bm -1: neither fits, or K keeps them off it).
GemmTile PickSmallTile(int M, int N, int K, int relay_rows)
{
    GemmTile best{-1, -1};
    double us = 1e30;
    for (int bm : {128, 64}) {
        const double t = relay_rows % bm == 0 ? SmallTileUs(bm, 1, M, N, K) : -1.0;
        if (t < 0.0 || t >= us) continue;
        us = t;
        best = {bm, 128};
    }
    return best;
}

// Estimated time (us) of whole rounds of one of the larger tiles over K: its
// time per 64-deep stage with the device full, one more per tile for its
// prologue and epilogue, 6 for the launch. Fitted to rounds of 56..64 stages
// (M 515..4096, N 4608..37888) and of 14; only the order of the candidates
// matters, and where rounds are many and full the card's power limit levels
// them (2048x37888x3584: 442..453 us whatever the tile).
struct TileCost {
    GemmTile tile;
    int per_cu;
    double stage;
};
constexpr TileCost kTileCosts[] = {
    {{256, 256}, 1, 1.25}, {{192, 256}, 1, 1.05}, {{256, 128}, 1, 0.72}, {{128, 256}, 1, 0.73}, {{128, 128}, 2, 1.02}};

double TileUs(const TileCost &c, int M, int N, int K)
{
    const int64_t tiles = int64_t((M + c.tile.bm - 1) / c.tile.bm) * ((N + c.tile.bn - 1) / c.tile.bn);
    const int64_t slots = int64_t(CuCount()) * c.per_cu;
    return 6.0 + double((tiles + slots - 1) / slots) * (K / kPipeK * c.stage + 1.0);
}

}  // namespace

GemmTile GemmPickTile(int M, int N, int relay_rows, bool coresident, int K)
{
    // No relay and K on the pipelined kernels: the cheapest by the estimates
    // above. Every tile runs the same MFMA and K order, so the choice never
    // changes the arithmetic. Measured against the rule below, which knows
    // neither K nor the tiles' rates: 515x24576x4096 177 -> 124 us,
    // 1500x24576x4096 299 -> 253, 3072x6144x4096 173 -> 152, 3072x9728x896
    // 79 -> 62, 2048x9728x896 59 -> 50.
    const GemmTile small = PickSmallTile(M, N, K, relay_rows);
    if (relay_rows == 0 && !coresident && K % kPipeK == 0 && !ForceSimple() && MainLoopMode() == 2) {
        GemmTile best = small;
        double us = small.bm > 0 ? SmallTileUs(small.bm, 1, M, N, K) : 1e30;
        for (const TileCost &c : kTileCosts) {
            const double t = TileUs(c, M, N, K);
            if (t >= us) continue;
            us = t;
            best = c.tile;
        }
        return best;
    }
    if (small.bm > 0) return small;
    return PickRelayTile(M, N, relay_rows, coresident);
}

// A small product whose cheapest row tile does not divide the relay tile (192
// or 576 rows in 128 row tiles): GemmSplitKernel in one piece, which releases
// any whole 64-row blocks (576x4096x4096, 64x256 tiles 61 us before).
bool OnePieceRelay(int M, int N, int K, int relay_rows, StreamKPlan &pl)
{
    if (relay_rows <= 0 || !SplitPubOk(M, relay_rows) || ForceSimple() || MainLoopMode() != 2) return false;
    const GemmTile t = PickSmallTile(M, N, K, 0);
    if (t.bm < 0 || relay_rows % t.bm == 0) return false;
    pl = StreamKPlan{};
    pl.bm = t.bm;
    pl.bn = t.bn;
    pl.nk = K / kPipeK;
    pl.tiles = pl.G = ((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    pl.pmax = 1;
    return true;
}

bool GemmNormRelayFits(int M, int N, int K, int rows_per_tile, bool streamk_ws, int dtype)
{
    if (AddRmsNormRowCpl(N) == 0 || rows_per_tile <= 0 || M % rows_per_tile != 0) return false;
    StreamKPlan skp;
    if (streamk_ws && !ForceSimple() && PlanStreamK(M, N, K, skp) && SplitPubOk(M, rows_per_tile) && SplitNormOk(skp))
        return NormRelayResident(dtype, skp.bm, skp.bn, M, N, K, rows_per_tile, skp.G);
    if (OnePieceRelay(M, N, K, rows_per_tile, skp) && std::getenv("KR_GEMM_TILE") == nullptr)
        return NormRelayResident(dtype, skp.bm, skp.bn, M, N, K, rows_per_tile, skp.G);
    GemmTile t = GemmPickTile(M, N, rows_per_tile, false, K);
    if (const char *e = std::getenv("KR_GEMM_TILE")) {
        int bm = 0, bn = 0;
        if (std::sscanf(e, "%dx%d", &bm, &bn) == 2 && rows_per_tile % bm == 0) t = {bm, bn};
    }
    if (t.bm <= 0 || t.bm == 192) t = {256, 256};
    return NormRelayResident(dtype, t.bm, t.bn, M, N, K, rows_per_tile, 0);
}

void GemmStreamKNeeds(int M, int N, int K, size_t *ws_bytes, int *counters)
{
    StreamKPlan pl;
    if (PlanStreamK(M, N, K, pl)) {
        *ws_bytes = pl.WsBytes();
        *counters = pl.tiles;
    } else {
        *ws_bytes = 0;
        *counters = 0;
    }
}

// Wave tail of a plain data-parallel 256x256 grid (the 8-wave staged kernel,
// no relay, no RoPE / norm / unary epilogue, no forced tile): when its tiles
// are not a whole number of rounds on the device, the last round runs partly
// idle (gate/up 2048x37888: 1184 tiles = 4 rounds + 160). Then the columns
// that fill whole rounds stay one launch (a), and the rest run as a second
// launch (b) of 192x256 tiles, one round of three-quarter tiles instead of a
// full round. Every tile shape runs the same MFMA over the same k16 chunks
// in the same order: the same bits. The SwiGLU epilogue splits with C (its
// gate/up groups of 8 never straddle a 256-column boundary).
// KR_GEMM_TAIL=0 keeps one launch.
bool SplitWaveTail(const GemmDesc &d, GemmDesc &a, GemmDesc &b)
{
    static const bool on = [] {
        const char *e = std::getenv("KR_GEMM_TAIL");
        return e == nullptr || std::atoi(e) != 0;
    }();
    if (!on || d.bm != 0 || d.bn != 0 || d.coresident || d.order_rows != 0) return false;
    if (d.pub.ctrl != nullptr || d.wait.ctrl != nullptr || d.tail_act != nullptr || d.y != nullptr ||
        d.rope_cos != nullptr || d.norm_y != nullptr)
        return false;
    if (d.K % kPipeK != 0 || ForceSimple() || MainLoopMode() != 2 || PipeWaves() != 8) return false;
    StreamKPlan skp;
    if (d.streamk && PlanStreamK(d.M, d.N, d.K, skp)) return false;
    const int64_t cus = CuCount();
    const int64_t tm = (d.M + 255) / 256, tn = (d.N + 255) / 256;
    const int64_t rounds = tm * tn / cus;
    if (rounds < 1 || (tm * tn) % cus == 0 || (rounds * cus) % tm != 0) return false;
    const int64_t n1 = rounds * cus / tm * 256;  // columns of the whole rounds
    const int64_t n2 = d.N - n1;
    if (n2 <= 0 || ((d.M + 191) / 192) * ((n2 + 255) / 256) > cus) return false;
    // against the cheapest single launch (the second launch runs as the first
    // drains: no launch time of its own)
    double us = 1e30;
    for (const TileCost &c : kTileCosts) us = std::min(us, TileUs(c, d.M, d.N, d.K));
    if (TileUs(kTileCosts[0], d.M, int(n1), d.K) + TileUs(kTileCosts[1], d.M, int(n2), d.K) - 6.0 >= us) return false;
    a = d;
    b = d;
    a.N = int(n1);
    a.bm = 256;
    a.bn = 256;
    b.N = int(n2);
    b.bm = 192;
    b.bn = 256;
    b.Bt = static_cast<const uint16_t *>(d.Bt) + n1 * d.ldb;
    if (d.C != nullptr) b.C = static_cast<uint16_t *>(d.C) + n1;
    if (d.bias != nullptr) b.bias = static_cast<const uint16_t *>(d.bias) + n1;
    if (d.epi_act != nullptr) b.epi_act = static_cast<uint16_t *>(d.epi_act) + n1 / 2;
    return true;
}

namespace {

// What a launch runs: a split plan (G > 0), or data-parallel tiles t.
struct Route {
    StreamKPlan split;
    GemmTile t{-1, -1};
};

Route RouteOf(const GemmDesc &d)
{
    const int relay_rows = d.pub.ctrl != nullptr ? d.pub.rows_per_tile : 0;
    GemmTile t = GemmPickTile(d.M, d.N, relay_rows, d.coresident, d.K);
    const char *forced = std::getenv("KR_GEMM_TILE");
    if (forced != nullptr) {
        // tile sweep override "BMxBN" (measurement aid; bits are unchanged)
        int bm = 0, bn = 0;
        if (std::sscanf(forced, "%dx%d", &bm, &bn) == 2 && (relay_rows == 0 || relay_rows % bm == 0)) t = {bm, bn};
    }
    if (d.bm > 0) {
        // a forced M tile pairs with the widest N tile built for it
        t.bm = d.bm;
        t.bn = d.bn > 0 ? d.bn : 256;
    } else if (d.bn > 0) {
        t.bn = d.bn;
    }
    if (t.bm < 0) throw std::runtime_error("gemm: relay tile rows must be a multiple of 64");
    // 192x256 runs only on the staged 8-wave kernel; elsewhere 256x256 (the
    // same MFMA and K order: the same bits)
    if (t.bm == 192 && (d.K % kPipeK != 0 || ForceSimple() || MainLoopMode() != 2 ||
                        d.tail_act != nullptr || d.pub.ctrl != nullptr || d.wait.ctrl != nullptr))
        t = {256, 256};
    Route r;
    r.t = d.epi_act == nullptr ? t : SwigluTile(t, LoopOf(t.bm, t.bn, d.M, d.N, d.K, RowSpan(d.lda, d.ldb), false, false));
    if (d.bm != 0 || d.bn != 0 || d.wait.ctrl != nullptr || d.tail_act != nullptr || d.epi_act != nullptr) return r;
    StreamKPlan pl;
    if (d.streamk && !ForceSimple() && PlanStreamK(d.M, d.N, d.K, pl) &&
        (d.pub.ctrl == nullptr || SplitPubOk(d.M, relay_rows)) && d.sk_ws != nullptr && d.sk_cnt != nullptr &&
        d.sk_ws_bytes >= pl.WsBytes() && d.sk_cnt_len >= pl.tiles && (d.norm_y == nullptr || SplitNormOk(pl))) {
        r.split = pl;
    } else if (forced == nullptr && d.order_rows == 0 && OnePieceRelay(d.M, d.N, d.K, relay_rows, pl)) {
        r.split = pl;
    }
    return r;
}

}  // namespace

void GemmLaunch(const GemmDesc &d, hipStream_t stream)
{
    if (d.K % 8 != 0) throw std::runtime_error("gemm: K must be a multiple of 8");
    if (d.M <= 0 || d.N <= 0 || d.K <= 0) throw std::runtime_error("gemm: empty shape");
    if ((reinterpret_cast<uintptr_t>(d.A) | reinterpret_cast<uintptr_t>(d.Bt)) & 15)
        throw std::runtime_error("gemm: A/Bt must be 16-byte aligned");
    if ((d.lda | d.ldb) % 8 != 0) throw std::runtime_error("gemm: lda/ldb must be multiples of 8");
    {
        GemmDesc a, b;
        if (SplitWaveTail(d, a, b)) {
            GemmLaunch(a, stream);
            GemmLaunch(b, stream);
            return;
        }
    }
    GemmParams p{};
    p.A = static_cast<const uint16_t *>(d.A);
    p.Bt = static_cast<const uint16_t *>(d.Bt);
    p.C = static_cast<uint16_t *>(d.C);
    p.bias = static_cast<const uint16_t *>(d.bias);
    p.lda = d.lda;
    p.ldb = d.ldb;
    p.ldc = d.ldc;
    p.M = d.M;
    p.N = d.N;
    p.K = d.K;
    p.pub = d.pub;
    p.wait = d.wait;
    p.store_kind = StoreKind();
    p.tail_act = static_cast<uint16_t *>(d.tail_act);
    p.tail_cols = d.tail_cols;
    p.epi_act = static_cast<uint16_t *>(d.epi_act);
    p.ld_act = d.ld_act;
    p.uy = d.y;
    p.uop = d.y_op;
    p.udt = d.y_dtype;
    p.ldy = d.ld_y > 0 ? d.ld_y : d.N;
    if (d.y != nullptr) {
        if (d.y_op != kEwGelu && d.y_op != kEwSilu && d.y_op != kEwCast)
            throw std::runtime_error("gemm: the unary consumer must be gelu, silu or cast");
        if (d.y_dtype != kBF16 && d.y_dtype != kF16 && d.y_dtype != kF32)
            throw std::runtime_error("gemm: unary consumer dtype");
        if (d.epi_act != nullptr || d.tail_act != nullptr || d.norm_y != nullptr || d.rope_cos != nullptr)
            throw std::runtime_error("gemm: one epilogue consumer per launch");
        if ((reinterpret_cast<uintptr_t>(d.y) & 15) != 0 || (p.ldy * int64_t(DTypeBytes(d.y_dtype))) % 16 != 0)
            throw std::runtime_error("gemm: unary consumer output must be 16-byte aligned rows");
    }
    if (d.rope_cos != nullptr) {
        if (d.rope_sin == nullptr || (d.rope_d != 64 && d.rope_d != 128) || d.rope_cols <= 0 ||
            d.rope_cols % d.rope_d != 0 || d.rope_cols > d.N || d.rope_pos0 < 0)
            throw std::runtime_error("gemm: RoPE epilogue needs cos/sin tables, head size 64 or 128, whole heads");
        if (p.epi_act != nullptr) throw std::runtime_error("gemm: RoPE and SwiGLU epilogues are exclusive");
        if ((reinterpret_cast<uintptr_t>(d.rope_cos) | reinterpret_cast<uintptr_t>(d.rope_sin)) & 15)
            throw std::runtime_error("gemm: RoPE tables must be 16-byte aligned");
        // every tile width is a multiple of 128, so tiles start on head boundaries
        p.rope_cos = static_cast<const uint16_t *>(d.rope_cos);
        p.rope_sin = static_cast<const uint16_t *>(d.rope_sin);
        p.rope_cols = d.rope_cols;
        p.rope_d = d.rope_d;
        p.rope_pos0 = d.rope_pos0;
    }
    if (p.epi_act != nullptr) {
        if (p.tail_act != nullptr) throw std::runtime_error("gemm: SwiGLU epilogue and tail consumer are exclusive");
        if (d.dtype != kBF16 && d.dtype != kF16) throw std::runtime_error("gemm swiglu: 16-bit output only");
        if (d.N % 16 != 0) throw std::runtime_error("gemm swiglu: N must be a multiple of 16 (gate/up groups of 8)");
        if ((reinterpret_cast<uintptr_t>(d.epi_act) & 15) || d.ld_act % 8 != 0 || d.ld_act < d.N / 2)
            throw std::runtime_error("gemm swiglu: act must be 16-byte aligned with ld_act >= N/2, a multiple of 8");
    }
    if (p.tail_act != nullptr) {
        if (p.pub.ctrl == nullptr || d.M % p.pub.rows_per_tile != 0)
            throw std::runtime_error("gemm tail: needs a relay release over whole tiles of M");
        if (d.dtype != kBF16 && d.dtype != kF16) throw std::runtime_error("gemm tail: 16-bit output only");
        if (d.N != 2 * d.tail_cols || d.ldc != d.N || d.tail_cols % 8 != 0)
            throw std::runtime_error("gemm tail: C must be a packed [M, 2*cols] interleaved gate/up buffer");
        if ((reinterpret_cast<uintptr_t>(d.C) | reinterpret_cast<uintptr_t>(d.tail_act)) & 15)
            throw std::runtime_error("gemm tail: buffers must be 16-byte aligned");
    }
    if (d.norm_y != nullptr) {
        if (d.pub.ctrl == nullptr || d.pub.rows_per_tile <= 0 || d.M % d.pub.rows_per_tile != 0)
            throw std::runtime_error("gemm add_rmsnorm: needs a relay release over whole tiles of M");
        if (d.norm_res == nullptr || d.norm_gamma == nullptr)
            throw std::runtime_error("gemm add_rmsnorm: residual and gamma are required");
        if (p.epi_act != nullptr || p.tail_act != nullptr || d.rope_cos != nullptr || d.order_rows != 0)
            throw std::runtime_error("gemm add_rmsnorm: excludes the SwiGLU epilogue/tail, RoPE and order_rows");
        if (d.ldc != d.N || AddRmsNormRowCpl(d.N) == 0)
            throw std::runtime_error("gemm add_rmsnorm: C must be packed (ldc == N) with N in 136..4096, N % 8 == 0");
        if ((reinterpret_cast<uintptr_t>(d.C) | reinterpret_cast<uintptr_t>(d.norm_res) |
             reinterpret_cast<uintptr_t>(d.norm_gamma) | reinterpret_cast<uintptr_t>(d.norm_y) |
             reinterpret_cast<uintptr_t>(d.norm_sum)) & 15)
            throw std::runtime_error("gemm add_rmsnorm: buffers must be 16-byte aligned");
        p.rn_res = static_cast<const uint16_t *>(d.norm_res);
        p.rn_gamma = static_cast<const uint16_t *>(d.norm_gamma);
        p.rn_y = static_cast<uint16_t *>(d.norm_y);
        p.rn_sum = static_cast<uint16_t *>(d.norm_sum);
        p.rn_rstd = d.norm_rstd;
        p.rn_eps = d.norm_eps;
        p.rn_cpl = AddRmsNormRowCpl(d.N);
        p.rn_spins = d.norm_max_spins > 0 ? d.norm_max_spins : kDefaultMaxSpins;
    }
    if (p.wait.ctrl != nullptr && p.wait.prod_rows <= 0) throw std::runtime_error("gemm: wait.prod_rows must be > 0");
    const Route route = RouteOf(d);
    const GemmTile t = route.t;
    const bool bf = d.dtype == kBF16;
    if (d.dtype != kBF16 && d.dtype != kF16) throw std::runtime_error("gemm: dtype must be bf16 or f16");
    const int order = d.order_rows;
    int tail = 0;
    if (d.tail_act != nullptr) {
        const int k = d.M / d.pub.rows_per_tile;
        tail = d.tail_tiles > 0 ? std::min(d.tail_tiles, k) : k;
    }
    if (route.split.G > 0) {
        const StreamKPlan &pl = route.split;
        if (pl.pmax > 1) {
            p.sk_ws = static_cast<float *>(d.sk_ws);
            p.sk_cnt = d.sk_cnt;
        }
        if (pl.bm == 128) {
            bf ? LaunchSplit<kBF16, 128, 128>(p, pl, stream) : LaunchSplit<kF16, 128, 128>(p, pl, stream);
        } else if (pl.bm == 64) {
            bf ? LaunchSplit<kBF16, 64, 128>(p, pl, stream) : LaunchSplit<kF16, 64, 128>(p, pl, stream);
        } else {
            bf ? LaunchTyped<kBF16, 256, 256>(p, 0, 0, stream, &pl) : LaunchTyped<kF16, 256, 256>(p, 0, 0, stream, &pl);
        }
        return;
    }
#define KR_GEMM_CASE(BM_, BN_)                                                                     \
    if (t.bm == BM_ && t.bn == BN_) {                                                              \
        bf ? LaunchTyped<kBF16, BM_, BN_>(p, order, tail, stream)                                  \
           : LaunchTyped<kF16, BM_, BN_>(p, order, tail, stream);                                  \
        return;                                                                                    \
    }
    KR_GEMM_CASE(256, 256)
    KR_GEMM_CASE(192, 256)
    KR_GEMM_CASE(256, 128)
    KR_GEMM_CASE(128, 256)
    KR_GEMM_CASE(128, 128)
    KR_GEMM_CASE(64, 128)
    KR_GEMM_CASE(64, 256)
#undef KR_GEMM_CASE
    throw std::runtime_error("gemm: unsupported tile " + std::to_string(t.bm) + "x" + std::to_string(t.bn));
}

}  // namespace kr

extern "C" int kr_gemm_route(int M, int N, int K, int64_t lda, int64_t ldb, int relay_rows, int ws, int use, int *bm,
                             int *bn, int *loop, int *pieces)
{
    using namespace kr;
    try {
        // stand-ins for device memory: the choice looks at their presence only
        static int32_t mark;
        GemmDesc d;
        d.M = M;
        d.N = N;
        d.K = K;
        d.lda = lda;
        d.ldb = ldb;
        if (relay_rows > 0) {
            d.pub.ctrl = &mark;
            d.pub.rows_per_tile = relay_rows;
        }
        if (use == 1) d.norm_y = &mark;
        if (use == 2) d.epi_act = &mark;
        size_t bytes = 0;
        int counters = 0;
        GemmStreamKNeeds(M, N, K, &bytes, &counters);
        if (ws != 0 && bytes > 0) {
            d.streamk = true;
            d.sk_ws = &mark;
            d.sk_ws_bytes = bytes;
            d.sk_cnt = &mark;
            d.sk_cnt_len = counters;
        }
        const Route r = RouteOf(d);
        const bool split = r.split.G > 0;
        *bm = split ? r.split.bm : r.t.bm;
        *bn = split ? r.split.bn : r.t.bn;
        *pieces = split ? r.split.pmax : 1;
        *loop = int(split && r.split.bm < 256 ? GemmLoop::kDeep
                                              : LoopOf(*bm, *bn, M, N, K, RowSpan(lda, ldb), split, use == 1));
        return 0;
    } catch (const std::exception &) {
        return 1;
    }
}
