// expert_i8_kernels.hip -- grouped expert GEMMs for few rows per expert (from a
// large decode batch to a prompt chunk) on int8 MFMA (gfx950), exact in f64.
//
// Semantics as the reference's mul_mat_id with Q8_0 activations
// (src/layers/moe.cpp:105-127, shared expert :161-165).  Per quant block b,
// v_mfma_i32_16x16x32_i8 gives the block's integer dots isum of 16 rows x 16
// weight columns; each term fp32(dw) * fp32(dx) * isum is exact in f64 and so is
// the sum of a row's terms, so the results equal the GEMVs' bit for bit: h needs
// no error bound and no fixup.
//
// What bounds it: at a few rows per expert every weight byte is used a few times
// only, so the weights' stream does, and each load's latency.  The GGUF rows of a
// wave's 32 columns are read 288 (Q4_0) or 272 (Q8_0) consecutive bytes per row
// and chunk, 16 bytes per lane, into registers a chunk ahead (9.2 or 8.7 KB per
// wave in flight, no padding rows, no chunk-major copy needed), and transposed to
// the MFMA operand through the wave's own LDS slab, which no barrier orders; the
// activations of a chunk, which a part's waves share, take two.  144-byte pieces
// of twice the columns ran at 3.6 instead of 4.2 TB/s.  The arithmetic is three
// f64 instructions per output and block (convert, scale by dw, fma by dx), each at
// an f32 instruction's rate on this chip, only for the groups of four rows that
// exist; two waves with half of a Q8_0 block of h each instead of one with all of
// it keep the workgroups short (the last round of them costs a workgroup's time).
// Measured, 35B-A3B shape, us: gate/up at 211 tokens Q4_0 217 (f16 path, GGUF rows)
// -> 79 (353 MB fetched, 4.5 TB/s; VALU issue is 49% of its cycles), down 84 -> 43;
// gate/up at 64 tokens 85 (streaming GEMV and the Q8_0 of h) -> 59; at 1000 tokens 161
// (2.9 TB/s, VALU issue 65%), down 84; at 512 tokens Q8_0 207 + 12 of fixups (f16 path
// with copies) -> 154, down 97 -> 78.
#include "qmoe_device.h"
#include "qmoe_internal.h"

#include <algorithm>
#include <type_traits>

namespace qmoe {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2i __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) uint8_t* GlobalBytes;
typedef const __attribute__((address_space(1))) u32x4a4* GlobalUnit;

// 64-value block pairs per chunk: 8 are 288 (Q4_0), 4 are 272 (Q8_0) consecutive
// bytes of a weight row.  The Q4_0 gate/up of 32 rows takes 4 (144 bytes): it is bound
// by its f64 steps, not by the stream, and three workgroups per CU hide more of them
// (prompt of 1000 tokens, 35B-A3B shape: 200 -> 187 us; the down GEMM, whose rows are
// one 8-pair chunk, lost: 91 -> 103).
constexpr int i8_pairs(int wt, bool gateup, int rows, int ks = 1) {
    return ks == 1 && wt == kTypeQ4_0 && !(gateup && rows == 32) ? 8 : 4;
}
// workgroups per CU: three where the registers of 16 rows, or of the short chunks, allow it
// (a split workgroup is launched where the grid does not fill the CUs: two waves per SIMD)
constexpr int i8_waves_per_simd(int wt, bool gateup, int rows, int ks) {
    return ks == 1 && (rows == 16 || (wt == kTypeQ4_0 && gateup)) ? 3 : 2;
}

// a workgroup of at most ROWS (16 or 32) rows of one expert, chunks of P pairs: a chunk's
// activation quants [pair][lane group][slot][16 bytes] and block scales [block][slot], padded
// against bank conflicts (a third of the gate/up's LDS cycles still conflict, with its LDS
// instructions 3 to 4% of the wave-cycles)
template <int ROWS> constexpr int kI8APair = 4 * ROWS * 16 + 16;
template <int ROWS> constexpr int kI8DBlock = ROWS + 4;
template <int P, int ROWS> constexpr int kI8ABytes = P * kI8APair<ROWS>;
template <int P, int ROWS> constexpr int kI8DBytes = 2 * P * kI8DBlock<ROWS> * 4;

template <int WT> constexpr int kI8PairBytes = 2 * BlockTraits<WT>::kBytes;
template <int WT, int P> constexpr int kI8RowBytes = P * kI8PairBytes<WT>;  // of a chunk
// LDS row stride: 36, 76 or 68 dwords
template <int WT, int P> constexpr int kI8Ld = kI8RowBytes<WT, P> + (kI8RowBytes<WT, P> == 288 ? 16 : 0);
template <int WT, int P> constexpr int kI8WBytes = 32 * kI8Ld<WT, P>;       // a wave's weight slab: 32 columns
template <int WT, int P, int ROWS, int CW>  // CW waves' weight slabs and their chunk's activations
constexpr int kI8PartBytes = CW * kI8WBytes<WT, P> + kI8ABytes<P, ROWS> + kI8DBytes<P, ROWS>;
template <int WT, int P, int ROWS, int CW, int KS>
constexpr size_t kI8LdsBytes = KS * (size_t)kI8PartBytes<WT, P, ROWS, CW> + 2 * 4 * ROWS * 4;

struct I8Args {
    int H, F, E;
    const uint8_t* w0; uint64_t w0_nb1, w0_nb2;  // gate (gate/up) or down
    const uint8_t* w1; uint64_t w1_nb1, w1_nb2;  // up
    const uint8_t* sh0; uint64_t sh0_nb1;        // shared gate or down
    const uint8_t* sh1; uint64_t sh1_nb1;        // shared up
    const int32_t* counters;                     // [1] n_tiles
    const int4* tiles;                           // {expert, first row, rows <= ROWS}
    int max_tiles;
    const int32_t* row_token;                    // gate/up: the token of each row
    const int8_t* a_qs; const float2* a_ds;      // activations: quants [rows][K], {scale, sum} [rows][K/32]
    int K, n_y, n_cg;                            // reduction length; column groups: workgroups x groups each
    int8_t* h_qs; float2* h_ds;                  // gate/up: the Q8_0 of h
    int act; const uint16_t* gelu_tab;
    float* ybuf;                                 // down: unweighted rows
};

// The slot of row r among a 16-row tile's MFMA rows: lane group g holds MFMA
// rows 4g .. 4g+3 of a column, so rows 4i .. 4i+3 sit at MFMA rows i, 4+i, 8+i,
// 12+i and a group of at most 4n rows needs only the first n results of a lane.
__device__ __forceinline__ int i8_slot(int r) { return (r & ~15) + 4 * (r & 3) + ((r & 15) >> 2); }

// One column's B operand of block J of a pair (this lane's 8 of the 32 quants)
// and its scale: pr = the column's pair in LDS.  Q4_0: 16 (q - 8), so the
// activations' scales carry a factor 1/16; k order {4g.., 16 + 4g..}.
template <int WT, int J> struct I8Block;
template <int J> struct I8Block<kTypeQ4_0, J> {
    uint32_t q0, q1, d;
    __device__ __forceinline__ void load(const uint32_t* pr, int g) {
        q0 = J == 0 ? pr[g] : pr[5 + g];
        q1 = J == 0 ? pr[g + 1] : 0u;
        d = J == 0 ? pr[0] : pr[4];
    }
    __device__ __forceinline__ long quants() const {
        const uint32_t u = J == 0 ? __builtin_amdgcn_alignbyte(q1, q0, 2) : q0;
        const uint32_t lo = ((u << 4) & 0xf0f0f0f0u) ^ 0x80808080u, hi = (u & 0xf0f0f0f0u) ^ 0x80808080u;
        return (long)(((uint64_t)hi << 32) | lo);
    }
    __device__ __forceinline__ float scale() const { return fp16_to_f32(J == 0 ? d : d >> 16); }
};
template <int J> struct I8Block<kTypeQ8_0, J> {
    uint32_t q0, q1, q2, d;
    __device__ __forceinline__ void load(const uint32_t* pr, int g) {
        const uint32_t* q = pr + 9 * J + 2 * g;
        q0 = q[0]; q1 = q[1];
        q2 = J == 0 ? q[2] : 0u;
        d = J == 0 ? pr[0] : pr[8];
    }
    __device__ __forceinline__ long quants() const {
        const uint32_t lo = J == 0 ? __builtin_amdgcn_alignbyte(q1, q0, 2) : q0;
        const uint32_t hi = J == 0 ? __builtin_amdgcn_alignbyte(q2, q1, 2) : q1;
        return (long)(((uint64_t)hi << 32) | lo);
    }
    __device__ __forceinline__ float scale() const { return fp16_to_f32(J == 0 ? d : d >> 16); }
};

// Orders this wave's LDS accesses before it with those after it, where lanes read what
// others of the wave wrote and no barrier stands between (the hardware keeps a wave's LDS
// operations in order: this keeps the compiler from moving them, and emits nothing).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// TAIL: the reduction length is not a multiple of a chunk, so a row's last chunk holds fewer pairs.
// KS: the workgroup's parts, each of CW waves (32 columns a wave) with slabs of its own; part p takes
// chunks p, p + KS, ... of the reduction.  The parts' f64 sums, exact and so the same in any order,
// meet in LDS before the epilogue.
template <int WT, bool GATEUP, int ROWS, bool TAIL, int CW, int KS>
__global__ __launch_bounds__(64 * CW * KS, i8_waves_per_simd(WT, GATEUP, ROWS, KS)) void k_expert_i8(I8Args a) {
    extern __shared__ __align__(16) uint8_t s_dyn[];
    static_assert(KS == 1 || GATEUP, "the down GEMM is not split");
    constexpr int kPairs = i8_pairs(WT, GATEUP, ROWS, KS);
    constexpr int kLd = kI8Ld<WT, kPairs>;
    constexpr int kPart = kI8PartBytes<WT, kPairs, ROWS, CW>;
    constexpr int kThreads = 64 * CW;  // of a part
    const int part = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / kThreads);
    uint8_t* s_part = s_dyn + part * kPart;
    uint8_t* s_a = s_part + CW * kI8WBytes<WT, kPairs>;
    float* s_d = (float*)(s_a + kI8ABytes<kPairs, ROWS>);
    float* s_amax = (float*)(s_dyn + KS * kPart);  // [CW waves][ROWS]
    int* s_sum = (int*)(s_amax + 4 * ROWS);
    // XCD-aware mapping (as the f16 GEMMs): XCD x takes every eighth tile, all column
    // groups of each; the shared expert's tiles, the fullest, come first.  The list
    // holds tiles with rows only: workgroups go to an XCD's four shader engines in
    // turn and hold a place for the microsecond that they take to find no rows
    // (with a workgroup per 16-row part of 128-row tiles, a third of the places).
    const int jb = (int)(blockIdx.x >> 3);
    const int tile_local = jb / a.n_y, y = jb - tile_local * a.n_y;
    const int tile_id = (int)(blockIdx.x & 7) + 8 * tile_local;
    const int4 tile = a.tiles[min(tile_id, a.max_tiles - 1)];  // (read along with the count)
    if (tile_id >= a.counters[1]) return;
    const int e = tile.x, p0 = tile.y, nr = tile.z;
    const bool sh = e >= a.E;
    const int tid = KS == 1 ? threadIdx.x : threadIdx.x & (kThreads - 1);  // within the part
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int col = lane & 15, g = lane >> 4;
    const int npairs = a.K >> 6, nblk = a.K >> 5;
    const int nchunk = (npairs + kPairs - 1) / kPairs;
    const int nstep = (nchunk + KS - 1) / KS;  // chunks per part; the last parts may have one fewer

    // this wave's 32 columns (two 16-column MFMA tiles): gate rows f0 .. f0 + 15 and
    // the same up rows, or down rows n0 .. n0 + 31.  Two waves share a Q8_0 block of h.
    // A down workgroup runs n_cg consecutive column groups (128 columns each); more than
    // one only where one chunk holds the activations: they are staged once, and the next
    // group's weights load while one is computed.
    const int ncg = GATEUP ? 1 : min(a.n_cg, (a.H >> 7) - y * a.n_cg);
    const int f0 = y * 16 * CW + 16 * wave, n0 = y * a.n_cg * 128 + 32 * wave;
    const uint32_t cs0 = (uint32_t)(sh ? a.sh0_nb1 : a.w0_nb1);
    const uint32_t cs1 = GATEUP ? (uint32_t)(sh ? a.sh1_nb1 : a.w1_nb1) : cs0;
    const uint8_t* wb0 = (sh ? a.sh0 : a.w0 + (uint64_t)e * a.w0_nb2) + (uint64_t)(GATEUP ? f0 : n0) * cs0;
    const uint8_t* wb1 = GATEUP ? (sh ? a.sh1 : a.w1 + (uint64_t)e * a.w1_nb2) + (uint64_t)f0 * cs1 : wb0 + (uint64_t)16 * cs0;
    // The wave's slab of a chunk is 32 kU units of 16 bytes: unit s = 64 i + lane is
    // bytes 16 (s % kU) .. of column s / kU's chunk (columns 16 .. from wb1); kL
    // loads per lane, the spare lanes of the last repeat the last unit
    constexpr int kU = kI8RowBytes<WT, kPairs> / 16;
    constexpr int kL = (32 * kU + 63) / 64;
    uint8_t* s_w = s_part + wave * kI8WBytes<WT, kPairs>;
    u32x4 wreg[kL];
    uint32_t woff[kL];
#pragma unroll
    for (int i = 0; i < kL; ++i) {
        const int s = min(64 * i + lane, 32 * kU - 1);
        const int r = s / kU, u = s - r * kU;
        woff[i] = (r < 16 ? (uint32_t)r * cs0 : (uint32_t)(r - 16) * cs1) + 16u * (uint32_t)u;
    }
    // this lane's unit of load i (the lane made opaque: hoisted out of the loop, what
    // is computed from it would take registers)
    auto unit_s = [&](int i) -> uint32_t {
        uint32_t l = (uint32_t)lane;
        asm volatile("" : "+v"(l));
        return 64 * i + 63 < 32 * kU ? 64 * i + l : min(64 * i + l, 32u * kU - 1u);
    };
    // a last chunk of np < kPairs pairs: a unit past its end moves back to end there
    // (dword-aligned), so nothing is read past a row
    auto unit_back = [&](uint32_t s, int np) -> uint32_t {
        return (uint32_t)max(0, 16 * (int)(s % kU) - (np * kI8PairBytes<WT> - 16));
    };
    // a uniform base made opaque: loads with a scalar base and one 32-bit offset per
    // lane, not a 64-bit running pointer per load
    auto base = [&](const uint8_t* w, int c) -> GlobalBytes {
        const uint64_t b = (uint64_t)(uintptr_t)w + (uint64_t)(c * kI8RowBytes<WT, kPairs>);
        return (GlobalBytes)(uintptr_t)(
            ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32) |
            (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b));
    };
    auto fetch = [&](int cg, int c) {
        const uint64_t skip = GATEUP ? 0 : (uint64_t)(128 * cg) * cs0;
        const GlobalBytes b0 = base(wb0 + skip, c), b1 = base(wb1 + skip, c);
        const int np = npairs - c * kPairs;
        const bool tail = TAIL && np < kPairs;
#pragma unroll
        for (int i = 0; i < kL; ++i) {
            uint32_t o = woff[i];
            asm volatile("" : "+v"(o));  // (its 64-bit extension kept out of registers too)
            if (tail) o -= unit_back(unit_s(i), np);
            if (64 * i + 63 < 16 * kU) wreg[i] = *(GlobalUnit)(b0 + o);
            else if (64 * i >= 16 * kU) wreg[i] = *(GlobalUnit)(b1 + o);
            else wreg[i] = *(GlobalUnit)((64 * i + lane < 16 * kU ? b0 : b1) + o);
        }
    };
    auto put = [&](int c) {
        const int np = npairs - c * kPairs;
#pragma unroll
        for (int i = 0; i < kL; ++i) {
            const uint32_t s = unit_s(i);
            uint8_t* d = s_w + 16 * s + (kLd - 16 * kU) * (s / kU);
            if (!TAIL || np >= kPairs) {
                *(u32x4*)d = wreg[i];
            } else {
                uint32_t* q = (uint32_t*)(d - unit_back(s, np));
                q[0] = wreg[i].x; q[1] = wreg[i].y; q[2] = wreg[i].z; q[3] = wreg[i].w;
            }
        }
    };
    if (KS == 1 || part < nchunk) fetch(0, part);

    // activations: thread t stages half-blocks of 16 values, half-block t % kHB of
    // rows t / kHB, + kThreads / kHB, ... of each chunk; even ones also the block's scale
    constexpr int kHB = 4 * kPairs, kRS = kThreads / kHB, kAR = ROWS / kRS;
    const int ahb = tid & (kHB - 1), ablk = ahb >> 1, ar0 = tid / kHB;
    uint32_t arow[kAR];
#pragma unroll
    for (int m = 0; m < kAR; ++m) {
        const int apos = p0 + min(kRS * m + ar0, nr - 1);  // rows past the group's repeat its last
        arow[m] = (uint32_t)(GATEUP ? a.row_token[apos] : apos);
    }
    u32x4 areg[kAR] = {};
    float dreg[kAR] = {};
    auto fetch_a = [&](int c) {
        if (TAIL && 2 * kPairs * c + ablk >= nblk) return;
#pragma unroll
        for (int m = 0; m < kAR; ++m) {
            if (m > 0 && nr <= kRS * m) break;
            uint32_t r = arow[m];
            asm volatile("" : "+v"(r));
            areg[m] = *(const u32x4*)(a.a_qs + (uint64_t)r * (uint32_t)a.K + (64 * kPairs * c + 16 * ahb));
            dreg[m] = a.a_ds[(uint64_t)r * (uint32_t)nblk + (2 * kPairs * c + ablk)].x;
        }
    };
    auto put_a = [&]() {
#pragma unroll
        for (int m = 0; m < kAR; ++m) {
            if (m > 0 && nr <= kRS * m) break;
            const int slot = i8_slot(kRS * m + ar0);
            // this half-block's part of each lane group's operand: Q4_0 {4g.., 16 + 4g..}: a
            // dword of each group's; Q8_0 {8g..}: two whole ones
            uint8_t* q = s_a + (ablk >> 1) * kI8APair<ROWS> + slot * 16 + 8 * (ablk & 1);
            if (WT == kTypeQ4_0) {
                uint32_t* q4 = (uint32_t*)(q + 4 * (ahb & 1));
                q4[0] = areg[m].x; q4[4 * ROWS] = areg[m].y; q4[8 * ROWS] = areg[m].z; q4[12 * ROWS] = areg[m].w;
            } else {
                uint8_t* q8 = q + (ahb & 1) * 2 * ROWS * 16;
                *(u32x2i*)q8 = u32x2i{areg[m].x, areg[m].y};
                *(u32x2i*)(q8 + ROWS * 16) = u32x2i{areg[m].z, areg[m].w};
            }
            if ((ahb & 1) == 0) s_d[ablk * kI8DBlock<ROWS> + slot] = WT == kTypeQ4_0 ? dreg[m] * 0.0625f : dreg[m];
        }
    };
    if (KS == 1 || part < nchunk) fetch_a(part);

    // the whole reduction and the epilogue for NQ groups of four rows
    auto run = [&](auto nq_c) {
        constexpr int NQ = decltype(nq_c)::value;
        constexpr int NM = (NQ + 3) / 4;  // 16-row MFMA tiles
        double acc[2][NQ];
        // one pair's operands
        struct Ops {
            u32x4 af[NM];
            I8Block<WT, 0> w0[2];
            I8Block<WT, 1> w1[2];
            float d[2][NQ];
        };
        auto load = [&](Ops& o, int pp) {
#pragma unroll
            for (int m = 0; m < NM; ++m)
                o.af[m] = *(const u32x4*)(s_a + pp * kI8APair<ROWS> + (g * ROWS + col + 16 * m) * 16);
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) {
                const uint32_t* pr = (const uint32_t*)(s_w + (16 * ct + col) * kLd + pp * kI8PairBytes<WT>);
                o.w0[ct].load(pr, g);
                o.w1[ct].load(pr, g);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < NQ; ++i) o.d[j][i] = s_d[(2 * pp + j) * kI8DBlock<ROWS> + 4 * g + 16 * (i >> 2) + (i & 3)];
        };
        auto block = [&](const Ops& o, auto j_c) {
            constexpr int J = decltype(j_c)::value;
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) {
                long bq;
                double dw;
                if constexpr (J == 0) { bq = o.w0[ct].quants(); dw = (double)o.w0[ct].scale(); }
                else { bq = o.w1[ct].quants(); dw = (double)o.w1[ct].scale(); }
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    const uint32_t x0 = J == 0 ? o.af[m].x : o.af[m].z, x1 = J == 0 ? o.af[m].y : o.af[m].w;
                    const v4i p = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(((uint64_t)x1 << 32) | x0), bq,
                                                                        v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (4 * m + i < NQ)
                            acc[ct][4 * m + i] =
                                __builtin_fma((double)p[i] * dw, (double)o.d[J][4 * m + i], acc[ct][4 * m + i]);
                }
            }
        };
        auto both = [&](const Ops& o) {
            block(o, std::integral_constant<int, 0>{});
            block(o, std::integral_constant<int, 1>{});
        };
        for (int cg = 0; cg < ncg; ++cg) {
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                for (int i = 0; i < NQ; ++i) acc[ct][i] = 0.0;
            if (cg > 0) wave_lds_order();  // (the group before's reads of the slab)
            for (int st = 0; st < nstep; ++st) {
                const int c = part + KS * st;
                const bool live = KS == 1 || c < nchunk;  // (uniform over the part)
                const bool stage = cg == 0;
                if (stage) {
                    if (st > 0) __syncthreads();  // the chunk before's activations are no longer read
                    if (live) put_a();
                }
                if (live) put(c);  // (the wave's own slab)
                if (stage) __syncthreads();
                else wave_lds_order();
                const bool last = c + KS >= nchunk;
                if (!last || cg + 1 < ncg) {  // (one place that fetches: two are twice the code)
                    fetch(last ? cg + 1 : cg, last ? 0 : c + KS);
                    if (nstep > 1) fetch_a(last ? 0 : c + KS);
                }
                const int np = !live ? 0 : TAIL ? min(kPairs, npairs - kPairs * c) : kPairs;
#pragma unroll 1
                for (int pp = 0; pp < np; ++pp) {
                    Ops o;
                    load(o, pp);
                    both(o);
                }
            }
            if (!GATEUP) {
#pragma unroll
                for (int i = 0; i < NQ; ++i) {
                    const int r = 4 * i + g;
                    if (r < nr) {
                        float* yr = a.ybuf + (uint64_t)(p0 + r) * a.H + (n0 + 128 * cg + col);
                        yr[0] = (float)acc[0][i];
                        yr[16] = (float)acc[1][i];
                    }
                }
            }
        }
        if (!GATEUP) return;
        if constexpr (KS > 1) {
            // over the slabs, which every wave is done with; part 0 then runs the epilogue
            static_assert((KS - 1) * (ROWS / 4) * 2 * kThreads * 8 <= KS * kPart, "the sums fit");
            double* red = (double*)s_dyn + tid;
            __syncthreads();
            if (part > 0)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                    for (int i = 0; i < NQ; ++i) red[kThreads * (2 * NQ * (part - 1) + NQ * ct + i)] = acc[ct][i];
            __syncthreads();
            if (part == 0)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                    for (int i = 0; i < NQ; ++i)
#pragma unroll
                        for (int p = 0; p < KS - 1; ++p) acc[ct][i] += red[kThreads * (2 * NQ * p + NQ * ct + i)];
        }
        // h and its Q8_0, as swiglu_q8_block32: the 16 lanes of a group hold half of
        // a row's 32-value block, the other wave of the pair the other half; the
        // block's amax and quant sum meet in LDS
        const int fb = y * (CW / 2) + (wave >> 1);
        float h[NQ];
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            h[i] = act_mul(a.act, a.gelu_tab, (float)acc[0][i], (float)acc[1][i]);
            float amax = __builtin_fabsf(h[i]);
            amax = dpp8_max<kDppQuadXor1>(amax);
            amax = dpp8_max<kDppQuadXor2>(amax);
            amax = dpp8_max<kDppRowHalfMirror>(amax);
            amax = dpp8_max<kDppRowMirror>(amax);
            if (col == 0 && part == 0) s_amax[wave * ROWS + 4 * i + g] = amax;
        }
        __syncthreads();
        float d[NQ];
        int sum[NQ];
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const int r = 4 * i + g;
            const float amax = fmaxf(s_amax[wave * ROWS + r], s_amax[(wave ^ 1) * ROWS + r]);
            d[i] = amax / 127.0f;
            const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
            const int q = (int)__builtin_rintf(h[i] * id);
            sum[i] = q;
            sum[i] = dpp8_add<kDppQuadXor1>(sum[i]);
            sum[i] = dpp8_add<kDppQuadXor2>(sum[i]);
            sum[i] = dpp8_add<kDppRowHalfMirror>(sum[i]);
            sum[i] = dpp8_add<kDppRowMirror>(sum[i]);
            if ((wave & 1) && col == 0 && part == 0) s_sum[wave * ROWS + r] = sum[i];
            if (r < nr && part == 0) a.h_qs[(uint64_t)(p0 + r) * a.F + f0 + col] = (int8_t)q;
        }
        __syncthreads();
        if (!(wave & 1) && col == 0 && part == 0) {
#pragma unroll
            for (int i = 0; i < NQ; ++i) {
                const int r = 4 * i + g;
                if (r < nr)
                    a.h_ds[(uint64_t)(p0 + r) * (a.F >> 5) + fb] =
                        make_float2(fp16_to_f32(f32_to_fp16(d[i])), __builtin_bit_cast(float, sum[i] + s_sum[(wave + 1) * ROWS + r]));
            }
        }
    };
    switch ((nr + 3) >> 2) {
        case 1: run(std::integral_constant<int, 1>{}); break;
        case 2: run(std::integral_constant<int, 2>{}); break;
        case 3: run(std::integral_constant<int, 3>{}); break;
        case 4: run(std::integral_constant<int, 4>{}); break;
        case 5: if constexpr (ROWS > 16) run(std::integral_constant<int, 5>{}); break;
        case 6: if constexpr (ROWS > 16) run(std::integral_constant<int, 6>{}); break;
        case 7: if constexpr (ROWS > 16) run(std::integral_constant<int, 7>{}); break;
        default: if constexpr (ROWS > 16) run(std::integral_constant<int, 8>{}); break;
    }
}

static I8Args base_i8_args(const LayerDesc& L, const Workspace& ws) {
    I8Args a{};
    a.H = L.H; a.F = L.F; a.E = L.E;
    a.counters = ws.counters;
    a.tiles = i8_tiles(ws);
    a.row_token = ws.row_token;
    a.h_qs = ws.hq_qs; a.h_ds = ws.hq_ds;
    a.ybuf = ws.ybuf;
    a.act = L.act;
    a.gelu_tab = L.gelu_tab;
    return a;
}

// 16 rows per workgroup (three workgroups per CU) at few rows per expert, 32 beyond, where 16
// would read the weights of most experts twice: from 14 rows in Q8_0 (two workgroups per CU), from
// 8 in Q4_0, whose 32-row gate/up fits three as well, except where the shared expert's full tiles,
// twice as long then, outlast a small grid (fewer than four workgroups per CU).  Layer us, 16 / 32:
// 35B-A3B Q4_0 139.8 / 141.0 at 5 rows, 162.6 / 154.4 at 8, 198.0 / 185.6 at 14; Gemma 4 135.9 /
// 139.3 at 4, 161.8 / 156.4 at 8; 128 experts of ffn 1536, hidden 4096 318.3 / 328.5 at 6, 345.7 /
// 345.8 at 8; 32 of ffn 512, hidden 2048 45.9 / 42.4 at 8, 53.1 / 48.1 at 11, with a shared expert
// 54.2 / 56.4 and 56.0 / 59.4; Q8_0 218.9 / 231.6 at 9, 254.8 / 249.2 at 14, Gemma 4 208.7 / 214.5
// at 10, 226.8 / 223.8 at 12.5.
int i8_tile_rows(const LayerDesc& L, int T) {
    const bool full_grid = (int64_t)L.E * (L.F / 64) >= 4 * (int64_t)L.n_cu;
    const int from = L.gu_type == kTypeQ4_0 && (!L.S || full_grid) ? 8 : 14;
    return (int64_t)T * L.K > from * (int64_t)L.E ? 32 : 16;
}

template <int WT, bool GATEUP, int ROWS, bool TAIL, int CW, int KS>
static hipError_t launch_i8_inst(const LayerDesc& L, int T, I8Args a, hipStream_t stream, hipEvent_t ev_start,
                                 hipEvent_t ev_stop) {
    const auto kern = k_expert_i8<WT, GATEUP, ROWS, TAIL, CW, KS>;
    constexpr size_t lds = kI8LdsBytes<WT, i8_pairs(WT, GATEUP, ROWS, KS), ROWS, CW, KS>;
    static_assert(lds <= 160 * 1024, "a CU's LDS");
    if constexpr (lds > 64 * 1024) {  // above the default dynamic LDS window: raise it (idempotent)
        const hipError_t err = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (err != hipSuccess) return err;
    }
    a.max_tiles = max_row_tiles(L, T, ROWS);
    const dim3 grid((unsigned)(8 * ((a.max_tiles + 7) / 8) * a.n_y));
    launch_timed(kern, grid, dim3(64 * CW * KS), lds, stream, ev_start, ev_stop, a);
    return hipGetLastError();
}

// A gate/up grid that leaves CUs idle (tiles go to the XCDs in turn: fewer than eight reach
// as many XCDs only) is bound by what one CU can fetch: workgroups of 32 ffn columns, two waves
// of them, each half of the reduction; below half the CUs four waves, each a quarter.  Layer us,
// whole workgroups / halves / quarters: 16 experts of ffn 512, hidden 1024, Q8_0, 64 tokens (184
// workgroups) 35.3 / 33.4 / 33.2; top-1 of 128 of ffn 512, hidden 2048, 17 tokens (152) 41.6 /
// 36.6 / 38.3; 64 of ffn 64, hidden 4096, 17 tokens (70) 64.3 / 53.8 / 51.4; 16 of ffn 128, hidden
// 4096, Q8_0, 13 tokens (32) 55.2 / 43.6 / 38.8; past the CUs' number level or slower (32 of ffn
// 1024, hidden 4096, 64 tokens, 736 workgroups 101.4 / 104.9 / 116.7).
static int i8_gateup_parts(const LayerDesc& L, int64_t tiles, int npairs) {
    const int64_t wgs = tiles * (L.F / 64), cus = (int64_t)L.n_cu * std::min<int64_t>(tiles, 8) / 8;
    if (2 * wgs <= cus && npairs >= 16) return 4;
    return wgs <= cus && npairs >= 8 ? 2 : 1;
}

template <int WT, bool GATEUP, int ROWS>
static hipError_t launch_i8_rows(const LayerDesc& L, int T, I8Args a, hipStream_t stream, hipEvent_t ev_start,
                                 hipEvent_t ev_stop) {
    const int npairs = a.K >> 6;
    if constexpr (GATEUP) {
        const int parts = i8_gateup_parts(L, max_row_tiles(L, T, ROWS), npairs);
        if (parts > 1) {
            a.n_y = L.F / 32;
            return parts == 4 ? launch_i8_inst<WT, true, ROWS, false, 2, 4>(L, T, a, stream, ev_start, ev_stop)
                              : launch_i8_inst<WT, true, ROWS, false, 2, 2>(L, T, a, stream, ev_start, ev_stop);
        }
    }
    // (n_embd is a multiple of 256: the gate/up's chunks of four pairs are whole)
    if constexpr (!GATEUP || i8_pairs(WT, GATEUP, ROWS) != 4)
        if (npairs % i8_pairs(WT, GATEUP, ROWS) != 0)
            return launch_i8_inst<WT, GATEUP, ROWS, true, 4, 1>(L, T, a, stream, ev_start, ev_stop);
    return launch_i8_inst<WT, GATEUP, ROWS, false, 4, 1>(L, T, a, stream, ev_start, ev_stop);
}

template <int WT, bool GATEUP>
static hipError_t launch_i8(const LayerDesc& L, int T, const I8Args& a, hipStream_t stream, hipEvent_t ev_start,
                            hipEvent_t ev_stop) {
    const bool wide = i8_tile_rows(L, T) == 32;
    return wide ? launch_i8_rows<WT, GATEUP, 32>(L, T, a, stream, ev_start, ev_stop)
                : launch_i8_rows<WT, GATEUP, 16>(L, T, a, stream, ev_start, ev_stop);
}

hipError_t launch_gateup_i8(const LayerDesc& L, const Workspace& ws, int T, hipStream_t stream, hipEvent_t ev_start,
                            hipEvent_t ev_stop) {
    I8Args a = base_i8_args(L, ws);
    a.w0 = L.w_gate; a.w0_nb1 = L.gate_nb1; a.w0_nb2 = L.gate_nb2;
    a.w1 = L.w_up; a.w1_nb1 = L.up_nb1; a.w1_nb2 = L.up_nb2;
    a.sh0 = L.w_sh_gate; a.sh0_nb1 = L.sh_gate_nb1;
    a.sh1 = L.w_sh_up; a.sh1_nb1 = L.sh_up_nb1;
    a.a_qs = ws.xq_qs; a.a_ds = ws.xq_ds;
    a.K = L.H;
    a.n_y = L.F / 64;
    a.n_cg = 1;
    return L.gu_type == kTypeQ4_0 ? launch_i8<kTypeQ4_0, true>(L, T, a, stream, ev_start, ev_stop)
                                  : launch_i8<kTypeQ8_0, true>(L, T, a, stream, ev_start, ev_stop);
}

hipError_t launch_down_i8(const LayerDesc& L, const Workspace& ws, int T, hipStream_t stream) {
    I8Args a = base_i8_args(L, ws);
    a.w0 = L.w_down; a.w0_nb1 = L.down_nb1; a.w0_nb2 = L.down_nb2;
    a.sh0 = L.w_sh_down; a.sh0_nb1 = L.sh_down_nb1;
    a.a_qs = ws.hq_qs; a.a_ds = ws.hq_ds;
    a.K = L.F;
    // Two column groups per workgroup save the second staging of its rows where one chunk
    // holds them and eight workgroups per CU are left (the kernel at 211 tokens, 35B-A3B Q4_0,
    // us: 45.5 with 1, 43.7 with 2, 46.5 with 4, 54.2 with 8).  Elsewhere they only halve the
    // grid.  Layer us, 2 / 1: 8 experts of ffn 4096, hidden 2048, 100 tokens 126.9 / 95.7; one
    // expert of ffn 4096, 32 tokens 122.8 / 92.0; 16 experts of ffn 512, hidden 1024, 64 tokens
    // 39.2 / 35.7; 35B-A3B Q8_0 (two chunks) at 100 tokens 193.5 / 185.6, Gemma 4 at 200 189.0 /
    // 183.8; one chunk: 35B-A3B Q4_0 at 450 tokens 184.7 / 189.3, top-1 of 128 experts at 300
    // 88.6 / 89.7 (2500 groups), top-4 of 32 at 100 61.9 / 60.6 (1000 groups).
    const int rows = i8_tile_rows(L, T);
    const bool one_chunk = (L.F >> 6) <= i8_pairs(L.dn_type, false, rows);
    const int64_t groups = (int64_t)max_row_tiles(L, T, rows) * (L.H / 128);
    a.n_cg = one_chunk && groups >= 8 * (int64_t)L.n_cu ? 2 : 1;
    a.n_y = (L.H / 128 + a.n_cg - 1) / a.n_cg;
    return L.dn_type == kTypeQ4_0 ? launch_i8<kTypeQ4_0, false>(L, T, a, stream, nullptr, nullptr)
                                  : launch_i8<kTypeQ8_0, false>(L, T, a, stream, nullptr, nullptr);
}

}  // namespace qmoe
