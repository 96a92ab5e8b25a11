// npu_weight_quant_batchmatmul, int8 weight stored [N, K] with one scale per column (what LinearWeightQuant keeps), or [K, N] where the
// estimates prefer it to weight_quant_gemm4.hip, more than 32 activation rows: a tiled GEMM on the 16-bit MFMA.
//
// A workgroup of eight wavefronts (4 x 2) owns 64 * WTM rows x 128 columns; a wavefront owns 16 * WTM x 64.  K is walked in stages
// of 64.  What bounds the kernel is the LDS (192 KiB of it pass per stage of a 256-row tile, at 85 bytes per clock; the MFMAs are busy
// half the time): a wavefront reads (WTM + 4) KiB of fragments per 4 * WTM MFMAs and every weight passes three times (raw bytes,
// image, fragment), so tall tiles pay where there are enough of them.
//   * activations: global -> LDS directly, three slots, two stages ahead;
//   * weights: raw bytes global -> LDS (three slots of 8 KiB), read back one stage before they are needed, converted to the exact
//     16-bit images of the integers between the MFMAs of the first half of a stage, and written to one of two image slots;
//   * fragments are double buffered in registers: those of the second half of a stage are requested before the MFMAs of the first,
//     those of the next stage before the MFMAs of the second, so no MFMA waits for its own operands;
//   * one barrier per stage, between its halves: by then every wavefront holds the fragments of the second half, so the stage's
//     activation and image slots are free.
// Measured against the general tiled kernel (one barrier per stage in front of all reads, tiles of 64 or 128 rows, K split by the tile
// count): 1024x11264x1664 fp16 74 -> 58.5 us, 509x7296x10368 bf16 177 -> 104, 1476x3072x3072 81 -> 51, 135x3968x2176 28 -> 18, 1.25
// times as fast on average over 120 shapes.  Two more forms, measured: raw bytes read as fragments and converted by every wavefront
// for itself (136 KiB per stage, but four times the conversions, which take issue slots from the MFMAs): the same to 5 % slower; with
// it tiles of 256 columns: 20 % slower.
// [K, N] weights (template parameter KN): a wavefront copies one k octet of all 128 columns and its lanes read the bytes of two columns
// each, row by row, so the images are written transposed; everything behind the images is the same.  The eight 2-byte reads make a
// stage 10 to 35 % longer than that of [N, K] (four 4-byte reads of a column quad with 8-byte image writes, conflict-free by a swizzle
// of their own, were no faster on tall tiles and 8 % slower on 128-row ones).  Before (weight_quant_gemm4.hip: 64 rows to a
// workgroup, every weight converted once per 64 rows) and now, us: 384x4096x11008 94 -> 65, 2048x4096x4096 99 -> 82, 700x2048x8192
// 51 -> 36, 145x10496x14560 112 -> 76, 100x14336x1040 36 -> 24, 44x4096x2816 21.5 -> 17; 0.85 of the time on average over 60 shapes.
// Rows are 128 bytes with the 16-byte chunks XOR-swizzled by the row pair (conflict-free fragment reads); a K that is not a multiple
// of 64 ends in a stage whose activations past K are loaded as zeros.
//     out[m, n] = scale[n] * (sum_k x[m, k] w[n, k] + offset[n] * X[m]) + bias[n]
// The row sums X[m] come from MFMAs against ones: wavefront column 0 takes the first half of every stage, column 1 the second.
// K may be split over S workgroups per tile: each publishes its float32 sums, the last arrival adds them in chunk order.
#include "weight_quant_common.h"
#include "weight_quant_kmajor_gemm.h"

namespace mi355 {
namespace {

struct WqKmGemmArgs {
    const uint16_t *x;
    const void *w;
    const uint16_t *scale, *offset, *bias;
    uint16_t *out;
    float *partial;                 // workspace [tile][chunk][wavefront][accumulator quad][lane] float32x4 (S > 1)
    uint32_t *counter;              // workspace [tile], zero on entry, left zero (S > 1)
    int64_t ldx, ldo;
    uint32_t ldw;
    int M, N, K;
    int tiles_m, tiles_n, items_per_xcd, S;
};

constexpr int kBN = 128, kStageK = 64;
constexpr int kPitch = 128;                                    // bytes per LDS tile row: 64 k of 16 bits
constexpr int kImageBytes = kBN * kPitch, kRawBytes = kBN * kStageK;

template <int ACT, int WTM, bool KN>
__global__ __launch_bounds__(512, 1) void wq_kmajor_gemm_kernel(const WqKmGemmArgs p)
{
    constexpr int NW = 8, WGN = 2, WTN = 4;
    constexpr int BM = 64 * WTM;
    constexpr int A_BYTES = BM * kPitch;
    constexpr int IMAGE_BASE = 3 * A_BYTES, RAW_BASE = IMAGE_BASE + 2 * kImageBytes;
    constexpr int LA = WTM;                                    // activation loads of a wavefront per stage
    extern __shared__ __attribute__((aligned(1024))) char lds[];

    // workgroup -> (K chunk, tile): every XCD gets a contiguous run of items, rows fastest and chunks slowest, so that what an L2
    // holds is one K range of all rows and of a few weight strips
    const int tiles = p.tiles_m * p.tiles_n;
    const int item = (blockIdx.x & 7) * p.items_per_xcd + (blockIdx.x >> 3);
    if (item >= tiles * p.S) return;
    const int chunk = item / tiles, tile = item - chunk * tiles;
    const int m0 = (tile % p.tiles_m) * BM;
    const int n0 = (tile / p.tiles_m) * kBN;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int stages = (p.K + kStageK - 1) / kStageK;
    const int s0 = (int)((int64_t)stages * chunk / p.S);       // first stage of this workgroup
    const int NSTG = (int)((int64_t)stages * (chunk + 1) / p.S) - s0;

    // ---- activations: a unit is 8 rows x 128 B.  Lane l fills LDS slot l: row l / 8, chunk slot l % 8, which must hold the row's
    // chunk (l % 8) ^ ((row >> 1) & 7); unit = i * 8 + wave, so (row >> 1) & 7 = 4 * (wave & 1) + (l / 8) / 2
    const int rows_a = min(BM, p.M - m0);
    const __amdgpu_buffer_rsrc_t rsrc_a =
        make_rsrc(p.x + (int64_t)m0 * p.ldx, (uint32_t)(((int64_t)(rows_a - 1) * p.ldx + p.K) * 2));
    const int rr = lane >> 3;
    const int k_lane = ((lane & 7) ^ (((wave & 1) << 2) | (rr >> 1))) * 8;      // first k of this lane's piece
    const uint32_t voff_a = (uint32_t)((rr * (int)p.ldx + k_lane) * 2);
    const uint32_t unit_stride_a = 16u * (uint32_t)p.ldx;
    const int k_left = p.K - s0 * kStageK - k_lane;            // a piece of stage s lies before the end of K if s * 64 < k_left
    // loads are never skipped: a stage past the end gets an out-of-range lane offset (zeros, no memory traffic)
    auto issue_a = [&](int s) {
        char *slot = lds + (s % 3) * A_BYTES;
        const uint32_t vo = s < NSTG && s * kStageK < k_left ? voff_a : kOutOfRange;
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int u = i * NW + wave;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_void *)(slot + u * 1024), 16, vo,
                                                     (uint32_t)u * unit_stride_a + (uint32_t)(s0 + s) * kPitch, 0, 0);
        }
    };

    // ---- weights: wavefront w copies the stage's 64 bytes of columns 16 w .. 16 w + 15; of a [K, N] weight rows 8 w .. 8 w + 7 (the
    // w-th k octet) of all 128 columns
    const int cols_valid = min(kBN, p.N - n0);
    const __amdgpu_buffer_rsrc_t rsrc_w =
        KN ? make_rsrc(static_cast<const char *>(p.w) + n0, (uint32_t)(p.K - 1) * p.ldw + (uint32_t)cols_valid)
           : make_rsrc(static_cast<const char *>(p.w) + (size_t)n0 * p.ldw, (uint32_t)(cols_valid - 1) * p.ldw + (uint32_t)p.K);
    const uint32_t voff_w = !KN ? (uint32_t)(lane >> 2) * p.ldw + (uint32_t)(lane & 3) * 16u
                            : (lane & 7) * 16 < cols_valid ? (uint32_t)(lane >> 3) * p.ldw + (uint32_t)(lane & 7) * 16u : kOutOfRange;
    auto issue_w = [&](int s) {
        const uint32_t so = KN ? (uint32_t)((s0 + s) * kStageK + wave * 8) * p.ldw : (uint32_t)wave * 16u * p.ldw + (uint32_t)(s0 + s) * 64u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (lds_void *)(lds + RAW_BASE + (s % 3) * kRawBytes + wave * 1024), 16,
                                                 s < NSTG ? voff_w : kOutOfRange, so, 0, 0);
    };
    // [N, K]: two runs of eight consecutive k of one column each: chunk c = t * 512 + wave * 64 + lane is k octet c % 8 of column c / 8.
    // [K, N]: a word per pair of rows of the octet with the bytes of columns 2 lane and 2 lane + 1 (run t is column 2 lane + t).
    u32x2 wx[2];
    auto read_raw = [&](int s) {
        const char *src = lds + RAW_BASE + (s % 3) * kRawBytes;
        if constexpr (KN) {
            typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int v = 0; v < 4; v++) {
                u16x2 rows;
                rows.x = *reinterpret_cast<const uint16_t *>(src + wave * 1024 + (2 * v) * 128 + lane * 2);
                rows.y = *reinterpret_cast<const uint16_t *>(src + wave * 1024 + (2 * v + 1) * 128 + lane * 2);
                wx[v >> 1][v & 1] = __builtin_bit_cast(uint32_t, rows);
            }
        } else {
#pragma unroll
            for (int t = 0; t < 2; t++) wx[t] = *reinterpret_cast<const u32x2 *>(src + (wave * 64 + lane) * 8 + t * 4096);
        }
    };
    auto expand = [&](int t, int s) {
        const int c = t * 512 + wave * 64 + lane, n = KN ? 2 * lane + t : c >> 3, o = KN ? wave : c & 7;
        u32x4 b;
        if constexpr (KN) {
#pragma unroll
            for (int v = 0; v < 4; v++) b[v] = sbytes_act2<ACT>(wx[v >> 1][v & 1], t, 2 + t);
        } else {
            const u32x2 lo = sbytes_act4<ACT>(wx[t][0]), hi = sbytes_act4<ACT>(wx[t][1]);
            b = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
        *reinterpret_cast<u32x4 *>(lds + IMAGE_BASE + (s & 1) * kImageBytes + n * kPitch + ((o ^ ((n >> 1) & 7)) * 16)) = b;
    };

    // ---- fragments: lane reads row lane % 16 of a 16-row tile, chunk ks * 4 + lane / 16, stored at slot chunk ^ ((row >> 1) & 7)
    const int frow = lane & 15;
    const int sw0 = ((lane >> 4) ^ ((frow >> 1) & 7)) * 16;
    const int a_off = (wm * WTM * 16 + frow) * kPitch;
    const int b_off = IMAGE_BASE + (wn * WTN * 16 + frow) * kPitch;
    u32x4 af[2][WTM], bf[2][WTN];
    auto read_frags = [&](int s, int ks) {
        const int sw = sw0 ^ (ks * 64);
        const char *sa = lds + (s % 3) * A_BYTES + a_off + sw, *sb = lds + (s & 1) * kImageBytes + b_off + sw;
#pragma unroll
        for (int j = 0; j < WTN; j++) bf[ks][j] = *reinterpret_cast<const u32x4 *>(sb + j * 16 * kPitch);
#pragma unroll
        for (int i = 0; i < WTM; i++) af[ks][i] = *reinterpret_cast<const u32x4 *>(sa + i * 16 * kPitch);
    };

    f32x4 P[WTM][WTN], xsum[WTM];
#pragma unroll
    for (int i = 0; i < WTM; i++) {
        xsum[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < WTN; j++) P[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const u32x4 ones = u32x4{kOnes2<ACT>, kOnes2<ACT>, kOnes2<ACT>, kOnes2<ACT>};
    const bool has_offset = p.offset != nullptr;
    auto row_sums = [&](int ks) {
        if (has_offset && wn == ks)
#pragma unroll
            for (int i = 0; i < WTM; i++) xsum[i] = mfma_act<ACT>(ones, af[ks][i], xsum[i]);
    };
    auto barrier = [&]() {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    issue_w(0);
    issue_w(1);
    issue_a(0);
    issue_a(1);
    issue_w(2);
    issue_a(2);
    wait_vmcnt<2 * LA + 1>();                                  // raw stages 0 and 1 and activation stage 0 have landed
    barrier();
    read_raw(0);
    expand(0, 0);
    expand(1, 0);
    read_raw(1);
    wait_lgkmcnt0();
    barrier();
    issue_w(3);
    read_frags(0, 0);
    // (a wait that the compiler counts: with a scalar load pending into the loop it would wait for all LDS reads of an iteration)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_sched_barrier(0);
    // in flight at the top of stage s: activations s + 1, raw s + 2, activations s + 2, raw s + 3, in this order; the fragments of
    // the first half and the raw bytes of stage s + 1 are in registers or on their way there
    for (int s = 0; s < NSTG; s++) {
        // Memory instructions are spread over the MFMAs: issued in a burst behind the barrier they wait for their queues, and the
        // MFMAs behind them with them.
        read_frags(s, 1);
#pragma unroll
        for (int j = 0; j < WTN; j++)
#pragma unroll
            for (int i = 0; i < WTM; i++) P[i][j] = mfma_act<ACT>(bf[0][j], af[0][i], P[i][j]);
        expand(0, s + 1);                                      // its slot was last read in stage s - 1
        expand(1, s + 1);
        constexpr int MF = WTM * WTN, RD = WTM + WTN, RAW = KN ? 8 : 1;   // MFMAs, fragment and raw reads of a half
        constexpr int R1 = MF >= 2 * RD ? 1 : 2;               // LDS reads per MFMA
#pragma unroll
        for (int q = 0; q < (RD + R1 - 1) / R1; q++) {
            __builtin_amdgcn_sched_group_barrier(0x100, R1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
#pragma unroll
        for (int q = 0; q < MF; q++) {
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        row_sums(0);
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<LA + 1>();                                  // activations s + 1 and raw s + 2 have landed
        wait_lgkmcnt0();                                       // the images of s + 1 are written, stage s is read
        barrier();
        read_frags(s + 1, 0);
        read_raw(s + 2);
        issue_a(s + 3);                                        // into the slots of activations s and raw s + 1
        issue_w(s + 4);
#pragma unroll
        for (int j = 0; j < WTN; j++)
#pragma unroll
            for (int i = 0; i < WTM; i++) P[i][j] = mfma_act<ACT>(bf[1][j], af[1][i], P[i][j]);
#pragma unroll
        for (int q = 0; q < (RD + RAW + R1 - 1) / R1; q++) {
            __builtin_amdgcn_sched_group_barrier(0x100, R1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
#pragma unroll
        for (int q = 0; q < LA + 1; q++) {
            __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, MF, 0);
        __builtin_amdgcn_sched_barrier(0);
        row_sums(1);
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the refills past the end (zeros) have landed
    __syncthreads();

    // ---- scales and offsets: acc[r] of the ones-MFMA is the sum of row lane % 16 for every r, so lanes 0 .. 15 publish component 0
    float *const xs = reinterpret_cast<float *>(lds);          // [wavefront column][row]
    if (lane < 16)
#pragma unroll
        for (int i = 0; i < WTM; i++) xs[wn * BM + wm * WTM * 16 + i * 16 + lane] = xsum[i][0];
    const int ncol0 = n0 + wn * WTN * 16 + (lane >> 4) * 4;    // tile j covers columns ncol0 + 16 j .. + 3 of this lane
    const __amdgpu_buffer_rsrc_t rsrc_s = make_rsrc(p.scale, (uint32_t)p.N * 2u);
    const __amdgpu_buffer_rsrc_t rsrc_o = make_rsrc(p.offset, has_offset ? (uint32_t)p.N * 2u : 0u);
    u32x2 sv[WTN], ov[WTN];
#pragma unroll
    for (int j = 0; j < WTN; j++) {
        sv[j] = __builtin_amdgcn_raw_buffer_load_b64(rsrc_s, (uint32_t)ncol0 * 2u + 32u * j, 0, 0);
        ov[j] = __builtin_amdgcn_raw_buffer_load_b64(rsrc_o, (uint32_t)ncol0 * 2u + 32u * j, 0, 0);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < WTM; i++) {
        const float *src = xs + wm * WTM * 16 + i * 16 + frow;
        const float X = src[0] + src[BM];
#pragma unroll
        for (int j = 0; j < WTN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float sc = (r & 1) ? act_hi<ACT>(sv[j][r >> 1]) : act_lo<ACT>(sv[j][r >> 1]);
                const float of = (r & 1) ? act_hi<ACT>(ov[j][r >> 1]) : act_lo<ACT>(ov[j][r >> 1]);
                P[i][j][r] = sc * __builtin_fmaf(of, X, P[i][j][r]);
            }
    }

    // ---- split K: publish, count, last arrival sums in chunk order
    if (p.S > 1) {
        constexpr int SC1 = 16;                                // cache-policy bit: agent scope
        constexpr uint32_t WAVE_BYTES = WTM * WTN * 64 * 16;
        constexpr uint32_t CHUNK_BYTES = NW * WAVE_BYTES;
        const __amdgpu_buffer_rsrc_t rsrc_p =
            make_rsrc(p.partial + (size_t)tile * p.S * (CHUNK_BYTES / 4), (uint32_t)p.S * CHUNK_BYTES);
        const uint32_t lane_off = (uint32_t)wave * WAVE_BYTES + (uint32_t)lane * 16u;
#pragma unroll
        for (int i = 0; i < WTM; i++)
#pragma unroll
            for (int j = 0; j < WTN; j++)
                buffer_store_b128<SC1>(__builtin_bit_cast(u32x4, P[i][j]), rsrc_p, lane_off + (i * WTN + j) * 1024, (uint32_t)chunk * CHUNK_BYTES);
        wait_vmcnt<0>();                                       // this wavefront's sums have reached the coherence point
        __syncthreads();
        int &is_last = *reinterpret_cast<int *>(lds);
        if (threadIdx.x == 0) {
            const uint32_t old = __hip_atomic_fetch_add(p.counter + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            is_last = old == (uint32_t)(p.S - 1);
        }
        __syncthreads();
        if (!is_last) return;
        // The chunks are added in their order, whatever the order of arrival.  Tiles of 128 rows and more take the own one from registers:
        // the last arrival reads up to 128 KiB per chunk with the chip idle around it (us before -> after, sums identical: 1024x11264x1664
        // [N, K] 57.8 -> 56.1, four chunks; [K, N] 414x4224x5376 41.8 -> 39.6, three).  64-row tiles read it back: 1 % slower
        // otherwise (135x3968x2176 17.6 -> 17.7, 100x14336x1040 23.2 -> 23.5).  Several chunks requested at once, the unwanted out of
        // range, cost more than they hide (384x4096x4096 29.3 -> 30.4).
        f32x4 sum[WTM][WTN];
#pragma unroll
        for (int i = 0; i < WTM; i++)
#pragma unroll
            for (int j = 0; j < WTN; j++) sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int ch = 0; ch < p.S; ch++) {
            if (WTM > 1 && ch == chunk) {
#pragma unroll
                for (int i = 0; i < WTM; i++)
#pragma unroll
                    for (int j = 0; j < WTN; j++) sum[i][j] = sum[i][j] + P[i][j];
                continue;
            }
            f32x4 v[WTM][WTN];
#pragma unroll
            for (int i = 0; i < WTM; i++)
#pragma unroll
                for (int j = 0; j < WTN; j++)
                    v[i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_p, lane_off + (i * WTN + j) * 1024,
                                                                                              (uint32_t)ch * CHUNK_BYTES, SC1));
#pragma unroll
            for (int i = 0; i < WTM; i++)
#pragma unroll
                for (int j = 0; j < WTN; j++) sum[i][j] = sum[i][j] + v[i][j];
        }
#pragma unroll
        for (int i = 0; i < WTM; i++)
#pragma unroll
            for (int j = 0; j < WTN; j++) P[i][j] = sum[i][j];
        if (threadIdx.x == 0) __hip_atomic_store(p.counter + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // ---- output: lane holds row lane % 16 of tile i, columns ncol0 + 16 j + r
    const bool out_vec = (p.ldo & 3) == 0 && aligned_dev(p.out, 8);
#pragma unroll
    for (int j = 0; j < WTN; j++) {
        const int n = ncol0 + j * 16;
        if (n >= p.N) continue;                                // N is a multiple of 8: a quad is valid as a whole
        f32x4 bv = f32x4{0.f, 0.f, 0.f, 0.f};
        if (p.bias) {
#pragma unroll
            for (int r = 0; r < 4; r++) bv[r] = act_1<ACT>(p.bias[n + r]);
        }
#pragma unroll
        for (int i = 0; i < WTM; i++) {
            const int m = m0 + wm * WTM * 16 + i * 16 + frow;
            if (m >= p.M) continue;
            const f32x4 v = P[i][j] + bv;
            uint16_t *o = p.out + (int64_t)m * p.ldo + n;
            if (out_vec) {
                u32x2 pk;
                pk.x = pack_act2<ACT>(v[0], v[1]);
                pk.y = pack_act2<ACT>(v[2], v[3]);
                *reinterpret_cast<u32x2 *>(o) = pk;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = (uint16_t)pack_act2<ACT>(v[r], 0.0f);
            }
        }
    }
}

template <int ACT, int WTM, bool KN>
int launch_tile(WqKmGemmArgs p, hipStream_t s)
{
    constexpr int lds_bytes = 3 * 64 * WTM * kPitch + 2 * kImageBytes + 3 * kRawBytes;
    static_assert(lds_bytes <= 160 * 1024, "LDS budget");
    auto kern = wq_kmajor_gemm_kernel<ACT, WTM, KN>;
    static int attr_status = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (attr_status != hipSuccess) return MI355_ERR_LAUNCH;
    hipLaunchKernelGGL(kern, dim3((unsigned)(8 * p.items_per_xcd)), dim3(512), lds_bytes, s, p);
    return check_launch();
}

template <int ACT, bool KN>
int launch_act(const WqKmGemmArgs &p, int wtm, hipStream_t s)
{
    return wtm == 1 ? launch_tile<ACT, 1, KN>(p, s) : wtm == 2 ? launch_tile<ACT, 2, KN>(p, s) : wtm == 3 ? launch_tile<ACT, 3, KN>(p, s) : launch_tile<ACT, 4, KN>(p, s);
}

} // namespace

// the rows of a tile are addressed with 32-bit buffer offsets: rows far apart (one token of every sequence of a [128, 1024, 4096]
// batch: a pitch of 4194304) rule out the tall tiles
static bool offsets_fit(int wtm, int64_t ldx) { return (uint64_t)(64 * wtm) * (uint64_t)ldx * 2 < (1ull << 31); }

bool wq_kmajor_gemm_accepts(int64_t M, int64_t N, int64_t K, int64_t group_size, int64_t ldw, int64_t ldx, const void *x, const void *w,
                            const void *scale, const void *offset, bool n_major)
{
    return M > 32 && M <= 0x7fffffff && (group_size == 0 || group_size == K) && K >= 128 && K % 8 == 0 && N % 8 == 0 && ldw % 4 == 0 &&
           (n_major ? ldw >= N && (uint64_t)K * (uint64_t)ldw < (1ull << 31) : ldw >= K && (uint64_t)N * (uint64_t)ldw < (1ull << 32)) && ldx % 8 == 0 &&
           offsets_fit(2, ldx) && (x == nullptr || aligned(x, 16)) && (w == nullptr || aligned(w, 4)) && (scale == nullptr || aligned(scale, 4)) &&
           (offset == nullptr || aligned(offset, 4)) && !knob(kKnobWqGemmOff);
}

WqKmGemmPlan make_wq_kmajor_gemm_plan(int64_t M, int64_t N, int64_t K, int64_t group_size, int64_t ldw, int64_t ldx, const void *x,
                                      const void *w, const void *scale, const void *offset, size_t room, bool n_major,
                                      bool own_chunk_counts)
{
    WqKmGemmPlan pl{};
    pl.n_major = n_major;
    pl.ok = wq_kmajor_gemm_accepts(M, N, K, group_size, ldw, ldx, x, w, scale, offset, n_major);
    if (!pl.ok) return pl;
    // The tile and the split of K with the smallest estimated time: what a launch costs around the loop, rounds of the workgroups
    // that are resident at once (one to a CU, two of the 64-row tiles), but no less than the weights take from memory or the tiles
    // through the L2; and for a split the exchange of the sums.  Fitted to every tile and split of 120 shapes, M = 33 .. 2048, K = 1024
    // .. 14336, N = 1024 .. 16384 spread evenly over their logarithms: the choice is 1.4 % behind the measured best on average.  [K, N]: the
    // stage times of 60 such shapes on operands that come from memory.  The collecting workgroup reads every chunk, of tiles of 128 rows and more
    // all but its own: over 94 further shapes of [N, K] and 125 of [K, N] the choice is 0.8 and 1.3 % behind (1.1 and 1.9 with the own one counted).
    constexpr double kBaseUs = 7.1;
    constexpr double kStageUsNk[5] = {0.41, 0.675, 0.515, 0.657, 0.762}, kStageUsKn[5] = {0.49, 0.75, 0.71, 0.87, 1.05};   // [0]: a 64-row tile alone on its CU
    const double *const kStageUs = n_major ? kStageUsKn : kStageUsNk;
    constexpr double kWeightBytesPerUs = 5.5e6, kL2BytesPerUs = 11.4e6, kExchangeUs = 2.2, kExchangeBytesPerUs = 7.5e6, kCollectorBytesPerUs = 100e3;
    const int64_t stages = (K + kStageK - 1) / kStageK;
    const int forced_bm = knob(kKnobWqgBm), forced_split = knob(kKnobWqgSplit);   // tuning aids
    const bool forced = forced_split >= 1 && forced_split <= stages && forced_split <= 16;
    double best = 1e300;
    for (int wtm = 1; wtm <= 4; wtm++) {
        if (forced_bm > 0 && forced_bm % 64 == 0 && forced_bm <= 256 && forced_bm != 64 * wtm) continue;
        if (!offsets_fit(wtm, ldx)) continue;
        const int64_t tiles = ((M + 64 * wtm - 1) / (64 * wtm)) * ((N + kBN - 1) / kBN);
        if (tiles > 0x7fffffff / 16) continue;
        for (int S = 1; S <= 16; S++) {
            const int64_t slots = wtm == 1 ? 2 * kNumCU : kNumCU, wgs = tiles * S;
            if (forced && S != forced_split) continue;
            if (!forced && S > 1 && (wgs > slots || stages / S < 4)) break;
            const int64_t chunk_bytes = 64 * wtm * kBN * 4;
            if (S > 1 && ((uint64_t)tiles * 4 > kWorkspaceCounterBytes || (uint64_t)(wgs * chunk_bytes) > ((uint64_t)128 << 20) ||
                          kWorkspaceZeroBytes + (uint64_t)(wgs * chunk_bytes) > room)) continue;
            double us = (double)((wgs + slots - 1) / slots * ((stages + S - 1) / S)) * kStageUs[wtm == 1 && wgs <= kNumCU ? 0 : wtm];
            const double mem = (double)K * (double)N / kWeightBytesPerUs, l2 = (double)tiles * (128 * wtm + kBN) * (double)K / kL2BytesPerUs;
            us = kBaseUs + (us > mem ? us > l2 ? us : l2 : mem > l2 ? mem : l2);
            if (S > 1) us += kExchangeUs + (double)(wgs * chunk_bytes) * 2.0 / kExchangeBytesPerUs + (double)((wtm > 1 && !own_chunk_counts ? S - 1 : S) * chunk_bytes) / kCollectorBytesPerUs;
            if (us < best) {
                best = us;
                pl.us = us;
                pl.wtm = wtm;
                pl.S = S;
                pl.partial_bytes = S > 1 ? (size_t)(wgs * chunk_bytes) : 0;
            }
        }
    }
    pl.counter_bytes = pl.S > 1 ? kWorkspaceZeroBytes : 0;
    pl.ok = pl.wtm > 0;
    return pl;
}

int launch_wq_kmajor_gemm(const WqKmGemmPlan &pl, const void *x, int act_f16, const void *w, const void *scale, const void *offset,
                          const void *bias, void *out, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldo,
                          void *workspace, void *stream)
{
    WqKmGemmArgs p{};
    p.x = static_cast<const uint16_t *>(x);
    p.w = w;
    p.scale = static_cast<const uint16_t *>(scale);
    p.offset = static_cast<const uint16_t *>(offset);
    p.bias = static_cast<const uint16_t *>(bias);
    p.out = static_cast<uint16_t *>(out);
    p.counter = pl.S > 1 ? static_cast<uint32_t *>(workspace) : nullptr;
    p.partial = pl.S > 1 ? reinterpret_cast<float *>(static_cast<char *>(workspace) + pl.counter_bytes) : nullptr;
    p.ldx = ldx;
    p.ldo = ldo;
    p.ldw = (uint32_t)ldw;
    p.M = (int)M;
    p.N = (int)N;
    p.K = (int)K;
    p.tiles_m = (int)((M + 64 * pl.wtm - 1) / (64 * pl.wtm));
    p.tiles_n = (int)((N + kBN - 1) / kBN);
    p.items_per_xcd = (p.tiles_m * p.tiles_n * pl.S + 7) / 8;
    p.S = pl.S;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (pl.n_major) return act_f16 ? launch_act<1, true>(p, pl.wtm, s) : launch_act<0, true>(p, pl.wtm, s);
    return act_f16 ? launch_act<1, false>(p, pl.wtm, s) : launch_act<0, false>(p, pl.wtm, s);
}

} // namespace mi355
