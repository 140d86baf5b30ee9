// pt_mlp.hip — MLP ensemble surrogate on gfx950 MFMA (include/pandemic/pt_surrogate.h).
//
// All matrix products run on v_mfma_f32_16x16x32_bf16: BF16 operands, FP32
// accumulation, K in ascending order.  Every launch covers all ensemble
// members, which train on the same batch.  A training step is ten launches:
//
//   forward, 5   bias + GELU in the epilogue; the first layer gathers its
//                rows of X itself, the last one goes on to the loss: output
//                gradients, their column sums and the squared errors
//   backward, 4  input gradients; GELU backward and the column sums in the
//                epilogue (the first also closes the step's loss)
//   update, 1    the weight gradients of all layers, each tile followed by
//                its Adam step in the epilogue
//
// The products are small (2.7 GFLOP for 5 members at batch 1024, 1 us of the
// chip's MFMA rate), so the loads' latency, the epilogues' traffic and the
// launches bound a step: 5 members x 1024, 395 -> 165 us per step (19 launches
// and the FP32 gradients' round trips before).
//
// MFMA lane layout (checked on the device): lane l supplies row l % 16 of A
// and column l % 16 of B with eight K values each (K group l / 16), and
// receives C[4 (l / 16) + r][l % 16], r = 0..3.
//
// GELU is the exact form x * Phi(x), Phi(x) = (1 + erf(x / sqrt 2)) / 2
// (Hendrycks and Gimpel, 2016), through the HIP device erff / expf.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/pandemic/pt_surrogate.h"
#include "pt_day.h"

using namespace pt;

namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kDims[PT_MLP_LAYERS + 1] = {PT_MLP_IN, PT_MLP_HIDDEN, PT_MLP_HIDDEN, PT_MLP_HIDDEN, PT_MLP_HIDDEN,
                                           PT_MLP_OUT};
constexpr int kTile = 64;      // rows and columns of a tile (the loss tiles: kColRows rows), K per step
constexpr int kGemmThreads = 256;
constexpr int kXcds = 8;
constexpr int kMaxWidth = PT_MLP_OUT;  // widest layer output
constexpr int64_t kSlotRows = 2048;    // result rows per pinned slot: 5.9 MB

// Offsets of W_l and b_l in a member's parameter block.
struct Layout {
    int64_t w[PT_MLP_LAYERS], b[PT_MLP_LAYERS], count;
    Layout() {
        int64_t o = 0;
        for (int l = 0; l < PT_MLP_LAYERS; ++l) {
            w[l] = o;
            o += (int64_t)kDims[l] * kDims[l + 1];
            b[l] = o;
            o += kDims[l + 1];
        }
        count = o;
    }
};

// 2 Phi(x); GELU and its derivative from it.
__device__ __forceinline__ float two_phi(float x) { return 1.0f + erff(x * 0.70710678118654752f); }
__device__ __forceinline__ float gelu(float x, float phi2) { return 0.5f * x * phi2; }
__device__ __forceinline__ float gelu_grad(float x, float phi2) {
    const float cdf = 0.5f * phi2;
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

// One operand of a tile's product, ROWS (rows of A or columns of B) x K.
// Stored with K contiguous (KMAJOR false: base[row * ld + k]) or with the
// rows contiguous (base[k * ld + row]); either way 64 K values of it are runs
// of 64 contiguous elements in memory, read by the whole block as 16-byte
// vectors (every stride, offset and extent here is a multiple of 8) and kept
// in LDS as they come, 128 bytes per run.  A K-contiguous fragment is one
// 16-byte LDS read per lane; a K-major one is two transposing reads
// (ds_read_b64_tr_b16: of 4 K rows x 16 columns, lane i of 16 receives column
// i).  Runs are placed so that the 16 lanes of a fragment spread over all
// banks: the 16-byte chunk index is XORed with the run's row.
//
// Rows past the operand's extent repeat its last one (their products are not
// stored); K past its extent is zeroed on the way to LDS.
template <bool KMAJOR, int ROWS>
struct Operand {
    static_assert(!KMAJOR || ROWS == kTile, "K-major operands come in 64-column tiles");
    static constexpr int V = (KMAJOR ? kTile : ROWS) * 8 / kGemmThreads;  // vectors per thread and K step
    const bf16* p;     // uniform; this thread's vectors are at 32-bit offsets
    int64_t ld;
    int K;
    uint32_t at[V];    // vectors of K step 0
    uint32_t back[V];  // and how far back the step's first K value is
    __device__ __forceinline__ Operand(const bf16* base, int64_t ld_, int extent, int row0, int K_)
        : p(base), ld(ld_), K(K_) {
        const int run = threadIdx.x >> 3, c = threadIdx.x & 7;
#pragma unroll
        for (int q = 0; q < V; ++q) {
            const int r = run + 32 * q;
            back[q] = KMAJOR ? (uint32_t)r * (uint32_t)ld : (uint32_t)c * 8;
            at[q] = back[q] + (KMAJOR ? (uint32_t)(row0 + (row0 + c * 8 < extent ? c * 8 : 0))
                                      : (uint32_t)min(row0 + r, extent - 1) * (uint32_t)ld);
        }
    }
    __device__ __forceinline__ void load(bf16x8 (&v)[V], int k0) const {
        const int run = threadIdx.x >> 3, c = threadIdx.x & 7;
        const bf16* pk = p + (KMAJOR ? k0 * ld : (int64_t)k0);
        if (k0 + kTile <= K) {
#pragma unroll
            for (int q = 0; q < V; ++q) v[q] = *reinterpret_cast<const bf16x8*>(pk + at[q]);
        } else {
#pragma unroll
            for (int q = 0; q < V; ++q) {
                const bool in = k0 + (KMAJOR ? run + 32 * q : c * 8) < K;
                v[q] = *reinterpret_cast<const bf16x8*>(pk + (in ? at[q] : at[q] - back[q]));
            }
        }
    }
    __device__ __forceinline__ void store(bf16* s, const bf16x8 (&v)[V], int k0) const {
        const int run = threadIdx.x >> 3, c = threadIdx.x & 7;
#pragma unroll
        for (int q = 0; q < V; ++q) {
            const int r = run + 32 * q;
            bf16x8 x = v[q];
            if (k0 + kTile > K) {
                if ((KMAJOR ? k0 + r : k0 + c * 8) >= K) x = (bf16x8)(bf16)0.0f;
            }
            *reinterpret_cast<bf16x8*>(s + place(r, c)) = x;
        }
    }
    // Element offset of chunk c of run r.
    static __device__ __forceinline__ int place(int r, int c) {
        if (KMAJOR) return ((r & 48) | ((r >> 3) & 1) | ((r & 7) << 1)) * kTile + (c ^ ((r & 3) << 1)) * 8;
        return r * kTile + (c ^ ((r >> 1) & 7)) * 8;
    }
    // The fragment of K values k .. k + 31 of the 16 rows from row0.
    static __device__ __forceinline__ bf16x8 fragment(const bf16* s, int row0, int k, int lane) {
        const int g = lane >> 4, i = lane & 15;
        if constexpr (KMAJOR) {
            typedef __attribute__((address_space(3))) bf16x4* lds4;
            const bf16* x = s + place(k + 8 * g + (i >> 2), row0 / 8 + ((i & 3) >> 1)) + (i & 1) * 4;
            const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4)x);
            const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4)(x + 8 * kTile));  // K + 4: 8 runs on
            return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        } else {
            return *reinterpret_cast<const bf16x8*>(s + place(row0 + i, k / 8 + g));
        }
    }
};

constexpr int kRowPad = kTile + 4;  // floats per row of an output tile in LDS
constexpr size_t tile_lds(int TM) { return (size_t)2 * (TM + kTile) * kTile * sizeof(bf16); }
static_assert(tile_lds(kTile) >= kTile * kRowPad * sizeof(float) && tile_lds(128) >= 128 * kRowPad * sizeof(float),
              "an output tile fits in the operands' LDS");

// acc = A * B over all of K for one TM x 64 tile; four waves, each
// (TM / 2) x 32.  One barrier per K step of 64: operands are double buffered
// in LDS and loaded two steps ahead into registers, so that a K of 512 pays
// the memory latency about once (with one step ahead, two barriers and K-major
// operands transposed in the registers of a single wave: 16-24 us per product
// of 2.7 GFLOP, now 12-14, of which GELU and the stores are half).  Ends with a barrier: LDS may be reused.
template <int TM, class OA, class OB>
__device__ __forceinline__ void tile_product(const OA& A, const OB& B, int K, bf16* s,
                                             floatx4 (&acc)[TM / 32][2]) {
    constexpr int MI = TM / 32;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * 32;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    bf16* const sa[2] = {s, s + (TM + kTile) * kTile};
    bf16* const sb[2] = {s + TM * kTile, s + (TM + kTile + TM) * kTile};
    bf16x8 ra[2][OA::V], rb[2][OB::V];
    A.load(ra[0], 0);
    B.load(rb[0], 0);
    if (kTile < K) {
        A.load(ra[1], kTile);
        B.load(rb[1], kTile);
    }
    A.store(sa[0], ra[0], 0);
    B.store(sb[0], rb[0], 0);
    if (2 * kTile < K) {
        A.load(ra[0], 2 * kTile);
        B.load(rb[0], 2 * kTile);
    }
    __syncthreads();
    for (int k0 = 0; k0 < K; k0 += 2 * kTile) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = k0 + h * kTile;
            if (k >= K) break;
            if (k + kTile < K) {
                A.store(sa[1 - h], ra[1 - h], k + kTile);
                B.store(sb[1 - h], rb[1 - h], k + kTile);
                if (k + 3 * kTile < K) {
                    A.load(ra[1 - h], k + 3 * kTile);
                    B.load(rb[1 - h], k + 3 * kTile);
                }
            }
#pragma unroll
            for (int kc = 0; kc < kTile; kc += 32) {
                bf16x8 b[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) b[j] = OB::fragment(sb[h], wn + j * 16, kc, lane);
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    const bf16x8 a = OA::fragment(sa[h], wm + i * 16, kc, lane);
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[j], acc[i][j], 0, 0, 0);
                }
            }
            __syncthreads();
        }
    }
}

// The tile in LDS, row by row, so that the epilogues read and write global
// memory as 256-byte runs (four columns per thread, 16 rows per turn).
template <int TM>
__device__ __forceinline__ void tile_to_rows(const floatx4 (&acc)[TM / 32][2], float (*sc)[kRowPad]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * 32;
#pragma unroll
    for (int i = 0; i < TM / 32; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[wm + i * 16 + 4 * (lane >> 4) + r][wn + j * 16 + (lane & 15)] = acc[i][j][r];
    __syncthreads();
}

__device__ __forceinline__ floatx4 load4(const float* p) { return *reinterpret_cast<const floatx4*>(p); }
__device__ __forceinline__ void store4(float* p, floatx4 v) { *reinterpret_cast<floatx4*>(p) = v; }
__device__ __forceinline__ void store4(bf16* p, floatx4 v) {
    bf16x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = (bf16)v[k];
    *reinterpret_cast<bf16x4*>(p) = o;
}

// Blocks go round the XCDs, each with an L2 of its own: XCD x works through
// the x-th eighth of the tiles, so that the tiles that share operand rows, and
// a member's weights, share an L2.  -1: no tile.
__device__ __forceinline__ int tile_of_block(int block, int tiles) {
    const int per = (tiles + kXcds - 1) / kXcds, t = (block % kXcds) * per + block / kXcds;
    return block / kXcds < per && t < tiles ? t : -1;
}
inline int blocks_for_tiles(int tiles) { return (tiles + kXcds - 1) / kXcds * kXcds; }

// Where a training batch's rows come from: row b of the batch is row
// rows[step * B + b] of X and Y (rows null: row b itself).
struct Batch {
    const float *X, *Y;
    const int32_t* rows;
    const int64_t* step;  // may be null: step 0
    __device__ __forceinline__ const int32_t* first(int B) const { return rows ? rows + (step ? step[0] * B : 0) : rows; }
};

// One layer forward, C = act * W + bias over M rows.
enum Forward : int { FWD_FIRST = 0, FWD_HIDDEN, FWD_OUT, FWD_LOSS };
struct ForwardArgs {
    const bf16* A;  // activations [M][K]; FWD_FIRST writes them (the batch in BF16)
    int64_t a_z;    // per-member stride in elements (0: shared by all members)
    const bf16* W;  // [K][N]
    const float* bias;
    int64_t param_z;
    int M, N, K, members;
    float* out;     // FWD_FIRST, FWD_HIDDEN (null: prediction): gelu'(pre-activations); FWD_OUT: outputs
    int64_t out_z;
    bf16* act;      // FWD_FIRST, FWD_HIDDEN: activations; FWD_LOSS: output gradients
    int64_t act_z;
    Batch batch;    // FWD_FIRST, FWD_LOSS
    bf16* xb;       // FWD_FIRST (may be null): the batch's inputs in BF16
    float* part;    // FWD_LOSS: squared errors per tile [member][tile]
    float* colpart; // FWD_LOSS: column sums [member][row chunk][N]
};

// Bias gradients: db[n] = sum over rows of dz[row][n], per member.  Partial
// sums per row chunk come with the gradients: 64-row tiles of the hidden
// layers, chunks of kColRows rows of the output layer (4 row groups, added in
// a fixed order); the update adds the chunks in order.  Every order is fixed,
// so the result does not depend on scheduling.
constexpr int kColGroups = 4, kColRows = 128;

template <int MODE>
__global__ __launch_bounds__(kGemmThreads, MODE == FWD_LOSS ? 3 : 4) void k_forward(ForwardArgs g) {
    constexpr int TM = MODE == FWD_LOSS ? kColRows : kTile;
    __shared__ __attribute__((aligned(16))) bf16 s[tile_lds(TM) / sizeof(bf16)];
    __shared__ float s_sum[kColGroups][kTile];
    const int tn = (g.N + kTile - 1) / kTile, tm = (g.M + TM - 1) / TM;
    const int t = tile_of_block(blockIdx.x, tn * tm * g.members);
    if (t < 0) return;
    const int z = t / (tn * tm), mt = t / tn % tm, m0 = mt * TM, n0 = t % tn * kTile;
    const int tid = threadIdx.x, lane = tid & 63;
    const Operand<true, kTile> B(g.W + z * g.param_z, g.N, g.N, n0, g.K);
    floatx4 acc[TM / 32][2];
    if constexpr (MODE == FWD_FIRST) {
        // K = 16: one MFMA per tile, its K past 16 zero; rows gathered from X
        // by 64 x 2 threads.
        typedef Operand<false, kTile> OA;
        bf16x8 rb[2];
        B.load(rb, 0);
        const int32_t* rows = g.batch.first(g.M);
        const int r = tid >> 2, c = tid & 3, m = min(m0 + r, g.M - 1);
        bf16x8 x = (bf16x8)(bf16)0.0f;
        if (c * 8 < PT_MLP_IN) {
            const float* src = g.batch.X + (int64_t)(rows ? rows[m] : m) * PT_MLP_IN + c * 8;
            const floatx4 lo = load4(src), hi = load4(src + 4);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                x[k] = (bf16)lo[k];
                x[k + 4] = (bf16)hi[k];
            }
            if (g.xb && z == 0 && n0 == 0 && m0 + r < g.M)
                *reinterpret_cast<bf16x8*>(g.xb + (int64_t)m * PT_MLP_IN + c * 8) = x;
        }
        *reinterpret_cast<bf16x8*>(s + OA::place(r, c)) = x;
        bf16* sb = s + kTile * kTile;
        B.store(sb, rb, 0);
        __syncthreads();
        const int wave = tid >> 6, wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    OA::fragment(s, wm + i * 16, 0, lane), Operand<true, kTile>::fragment(sb, wn + j * 16, 0, lane),
                    floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        __syncthreads();
    } else {
        const Operand<false, TM> A(g.A + z * g.a_z, g.K, g.M, m0, g.K);
        tile_product<TM>(A, B, g.K, s, acc);
    }
    float(*sc)[kRowPad] = reinterpret_cast<float(*)[kRowPad]>(s);
    tile_to_rows<TM>(acc, sc);
    const int c4 = (tid & 15) * 4, col = n0 + c4;
    const bool in = col < g.N;
    const floatx4 bias = in ? load4(g.bias + z * g.param_z + col) : floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (MODE != FWD_LOSS) {
#pragma unroll
        for (int q = 0; q < TM / 16; ++q) {
            const int r = q * 16 + (tid >> 4), row = m0 + r;
            if (!in || row >= g.M) continue;
            const int64_t o = (int64_t)row * g.N + col;
            floatx4 pre = load4(&sc[r][c4]) + bias;
            if (MODE != FWD_OUT) {
                floatx4 a, phi2;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    phi2[k] = two_phi(pre[k]);
                    a[k] = gelu(pre[k], phi2[k]);
                }
                store4(g.act + z * g.act_z + o, a);
                if (!g.out) continue;
#pragma unroll
                for (int k = 0; k < 4; ++k) pre[k] = gelu_grad(pre[k], phi2[k]);
            }
            store4(g.out + z * g.out_z + o, pre);
        }
    } else {
        // Mean-squared error: dz = 2 (pred - y) / (M * N), in BF16 for the
        // products and in FP32 for the column sums.
        const int32_t* rows = g.batch.first(g.M);
        const float scale = 2.0f / (float)((int64_t)g.M * g.N);
        float e = 0.f;
#pragma unroll
        for (int q = 0; q < TM / 16; ++q) {
            const int r = q * 16 + (tid >> 4), row = m0 + r;
            if (!in || row >= g.M) continue;
            const floatx4 pred = load4(&sc[r][c4]) + bias;
            const floatx4 y = load4(g.batch.Y + (int64_t)(rows ? rows[row] : row) * g.N + col);
            floatx4 dz;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float d = pred[k] - y[k];
                e += d * d;
                dz[k] = d * scale;
            }
            store4(g.act + z * g.act_z + (int64_t)row * g.N + col, dz);
            store4(&sc[r][c4], dz);
        }
#pragma unroll
        for (int x = 32; x; x >>= 1) e += __shfl_xor(e, x, 64);
        __shared__ float s_e[kGemmThreads / 64];
        if (lane == 0) s_e[tid >> 6] = e;
        __syncthreads();
        const int c = tid % kTile, grp = tid / kTile, rn = min(TM, g.M - m0);
        float sum = 0.f;
        for (int r = grp; r < rn; r += kColGroups) sum += sc[r][c];
        s_sum[grp][c] = sum;
        __syncthreads();
        if (tid == 0) g.part[(z * tm + mt) * tn + n0 / kTile] = s_e[0] + s_e[1] + s_e[2] + s_e[3];
        if (grp == 0 && n0 + c < g.N) {
            float tot = 0.f;
#pragma unroll
            for (int q = 0; q < kColGroups; ++q) tot += s_sum[q][c];
            g.colpart[((int64_t)z * tm + mt) * g.N + n0 + c] = tot;
        }
    }
}

// The loss of every member from its tiles' squared errors, in a fixed order,
// by one block; then the step index advances, and the bias corrections
// 1 - beta^t of the Adam step that follows, t = Adam steps taken before this
// one + 1, are set.
struct StepArgs {
    const float* part;
    int tiles, members;  // tiles per member
    int64_t n;           // outputs per member
    float* loss;
    int64_t loss_z;
    int64_t* step;       // null: one loss per member, no Adam step; [0] step of the call, [1] Adam steps before the call
    float* bias_corr;    // [2]
};
__device__ __forceinline__ void finish_loss(const StepArgs& a) {
    const int lane = threadIdx.x & 63;
    const int64_t at = a.step ? a.step[0] : 0;
    for (int z = threadIdx.x >> 6; z < a.members; z += kGemmThreads / 64) {
        float t = 0.f;
        for (int b = lane; b < a.tiles; b += 64) t += a.part[z * a.tiles + b];
#pragma unroll
        for (int x = 32; x; x >>= 1) t += __shfl_xor(t, x, 64);
        if (lane == 0) a.loss[z * a.loss_z + at] = t / (float)a.n;
    }
    __syncthreads();
    if (threadIdx.x == 0 && a.step) {
        const double t = (double)(a.step[1] + at + 1);
        a.bias_corr[0] = (float)(1.0 - pow(0.9, t));
        a.bias_corr[1] = (float)(1.0 - pow(0.999, t));
        a.step[0] = at + 1;
    }
}

// Input gradients of a layer: dz_in = (dz W^T) * slope, M rows, N = the
// layer's inputs, K = its outputs; and their column sums per 64-row tile,
// colpart[member][row tile][N].  finish (the first of the chain): the block
// after the tiles closes the loss.
struct BackwardArgs {
    const bf16* dz;
    int64_t dz_z;
    const bf16* W;  // [N][K]
    int64_t param_z;
    int M, N, K, members;
    const float* slope;  // gelu'(pre-activations), from the forward pass (which has the erf at hand)
    int64_t slope_z;
    bf16* out;
    int64_t out_z;
    float* colpart;
    int finish;
    StepArgs step;
};
__global__ __launch_bounds__(kGemmThreads, 4) void k_backward(BackwardArgs g) {
    __shared__ __attribute__((aligned(16))) bf16 s[tile_lds(kTile) / sizeof(bf16)];
    __shared__ float s_cs[2][kTile];
    const int tn = (g.N + kTile - 1) / kTile, tm = (g.M + kTile - 1) / kTile, tiles = tn * tm * g.members;
    if (g.finish) {
        if (blockIdx.x == gridDim.x - 1) return finish_loss(g.step);
    }
    const int t = tile_of_block(blockIdx.x, tiles);
    if (t < 0) return;
    const int z = t / (tn * tm), mt = t / tn % tm, m0 = mt * kTile, n0 = t % tn * kTile;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const int c4 = (tid & 15) * 4, col = n0 + c4;
    // (M and N are multiples of 64 here: batches and hidden layers)
    floatx4 slope[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        slope[q] = load4(g.slope + z * g.slope_z + (int64_t)(m0 + q * 16 + (tid >> 4)) * g.N + col);
    const Operand<false, kTile> A(g.dz + z * g.dz_z, g.K, g.M, m0, g.K), B(g.W + z * g.param_z, g.K, g.N, n0, g.K);
    floatx4 acc[2][2];
    tile_product<kTile>(A, B, g.K, s, acc);
    float(*sc)[kRowPad] = reinterpret_cast<float(*)[kRowPad]>(s);
#pragma unroll
    for (int q = 0; q < 4; ++q) store4(&sc[q * 16 + (tid >> 4)][c4], slope[q]);
    __syncthreads();
    // Column sums of the tile: this lane's 8 rows, then the 4 lane groups of
    // a 16-column slice, then the two row halves, in that fixed order.
    float cs[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float* x = &sc[wm + i * 16 + 4 * (lane >> 4) + r][wn + j * 16 + (lane & 15)];
                const float d = acc[i][j][r] * *x;
                *x = d;
                cs[j] += d;
            }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        cs[j] += __shfl_xor(cs[j], 16, 64);
        cs[j] += __shfl_xor(cs[j], 32, 64);
        if (lane < 16) s_cs[wm / 32][wn + j * 16 + lane] = cs[j];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = q * 16 + (tid >> 4);
        store4(g.out + z * g.out_z + (int64_t)(m0 + r) * g.N + col, load4(&sc[r][c4]));
    }
    if (tid < kTile) g.colpart[((int64_t)z * tm + mt) * g.N + n0 + tid] = s_cs[0][tid] + s_cs[1][tid];
}

// Adam on one FP32 master parameter.
__device__ __forceinline__ void adam(float& p, float& m1, float& m2, float gi, float lr, float bc1, float bc2) {
    const float a = 0.9f * m1 + 0.1f * gi;
    const float b = 0.999f * m2 + 0.001f * gi * gi;
    m1 = a;
    m2 = b;
    const float mh = a / bc1, vh = b / bc2;
    p = p - lr * mh / (sqrtf(vh) + 1e-8f);
}

// Weight and bias gradients of every layer, dW = act^T dz over the batch and
// the column sums' totals: stored (ADAM false), or used at once for the Adam
// step of the tile's parameters, which saves the gradients' round trip.  Bound
// by memory: the parameters' 26 bytes each and the operands, 200 MB in 44 us
// for 5 members at batch 1024.  Blocks: the layers' tiles
// member by member, then 256 biases per block.
struct UpdateArgs {
    const bf16* act[PT_MLP_LAYERS];
    int64_t act_z[PT_MLP_LAYERS];
    const bf16* dz[PT_MLP_LAYERS];
    int64_t dz_z[PT_MLP_LAYERS];
    const float* colpart[PT_MLP_LAYERS];  // [member][R][width]
    int R_hidden, R_out;
    int members, batch;
    int64_t count;                        // parameters per member
    float* grads;
    float *p, *m1, *m2;
    bf16* pb;
    float lr;
    const float* bias_corr;
};
constexpr int layer_tiles(int l) { return (kDims[l] + kTile - 1) / kTile * ((kDims[l + 1] + kTile - 1) / kTile); }
constexpr int member_tiles() {
    int n = 0;
    for (int l = 0; l < PT_MLP_LAYERS; ++l) n += layer_tiles(l);
    return n;
}
constexpr int member_biases() {
    int n = 0;
    for (int l = 0; l < PT_MLP_LAYERS; ++l) n += kDims[l + 1];
    return n;
}
constexpr int kBiasBlocks = (member_biases() + kGemmThreads - 1) / kGemmThreads;

template <bool ADAM>
__global__ __launch_bounds__(kGemmThreads, 4) void k_update(UpdateArgs g) {
    __shared__ __attribute__((aligned(16))) bf16 s[tile_lds(kTile) / sizeof(bf16)];
    const int tid = threadIdx.x, tiles = member_tiles() * g.members;
    float bc1 = 0.f, bc2 = 0.f;
    if (ADAM) {
        bc1 = g.bias_corr[0];
        bc2 = g.bias_corr[1];
    }
    const int tile_blocks = (tiles + kXcds - 1) / kXcds * kXcds;
    if ((int)blockIdx.x >= tile_blocks) {
        const int b = blockIdx.x - tile_blocks, z = b / kBiasBlocks;
        int j = b % kBiasBlocks * kGemmThreads + tid;
        int64_t at = z * g.count;
#pragma unroll
        for (int l = 0; l < PT_MLP_LAYERS; ++l) {
            const int n = kDims[l + 1];
            at += (int64_t)kDims[l] * n;
            if (j >= 0 && j < n) {
                const int R = l == PT_MLP_LAYERS - 1 ? g.R_out : g.R_hidden;
                const float* c = g.colpart[l] + (int64_t)z * R * n + j;
                float sum = 0.f;
                for (int r = 0; r < R; ++r) sum += c[(int64_t)r * n];
                const int64_t i = at + j;
                if (ADAM) {
                    float p = g.p[i], m1 = g.m1[i], m2 = g.m2[i];
                    adam(p, m1, m2, sum, g.lr, bc1, bc2);
                    g.m1[i] = m1;
                    g.m2[i] = m2;
                    g.p[i] = p;
                    g.pb[i] = (bf16)p;
                } else {
                    g.grads[i] = sum;
                }
            }
            j -= n;
            at += n;
        }
        return;
    }
    const int t = tile_of_block(blockIdx.x, tiles);
    if (t < 0) return;
    const int z = t / member_tiles();
    int tl = t % member_tiles(), M = 0, N = 0;
    int64_t at = z * g.count, act_z = 0, dz_z = 0;
    const bf16 *act = nullptr, *dz = nullptr;
    bool found = false;
#pragma unroll
    for (int l = 0; l < PT_MLP_LAYERS; ++l) {
        if (found) continue;
        M = kDims[l];
        N = kDims[l + 1];
        act = g.act[l];
        act_z = g.act_z[l];
        dz = g.dz[l];
        dz_z = g.dz_z[l];
        if (tl < layer_tiles(l)) {
            found = true;
        } else {
            tl -= layer_tiles(l);
            at += (int64_t)M * N + N;
        }
    }
    const int tn = (N + kTile - 1) / kTile, m0 = tl / tn * kTile, n0 = tl % tn * kTile;
    const Operand<true, kTile> A(act + z * act_z, M, M, m0, g.batch), B(dz + z * dz_z, N, N, n0, g.batch);
    floatx4 acc[2][2];
    tile_product<kTile>(A, B, g.batch, s, acc);
    const int c4 = (tid & 15) * 4, col = n0 + c4;
    floatx4 p[4], m1[4], m2[4];
    if (ADAM) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = m0 + q * 16 + (tid >> 4);
            if (row >= M || col >= N) continue;
            const int64_t i = at + (int64_t)row * N + col;
            p[q] = load4(g.p + i);
            m1[q] = load4(g.m1 + i);
            m2[q] = load4(g.m2 + i);
        }
    }
    float(*sc)[kRowPad] = reinterpret_cast<float(*)[kRowPad]>(s);
    tile_to_rows<kTile>(acc, sc);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = q * 16 + (tid >> 4), row = m0 + r;
        if (row >= M || col >= N) continue;
        const int64_t i = at + (int64_t)row * N + col;
        const floatx4 gi = load4(&sc[r][c4]);
        if (ADAM) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float pk = p[q][k], m1k = m1[q][k], m2k = m2[q][k];
                adam(pk, m1k, m2k, gi[k], g.lr, bc1, bc2);
                p[q][k] = pk;
                m1[q][k] = m1k;
                m2[q][k] = m2k;
            }
            store4(g.m1 + i, m1[q]);
            store4(g.m2 + i, m2[q]);
            store4(g.p + i, p[q]);
            store4(g.pb + i, p[q]);
        } else {
            store4(g.grads + i, gi);
        }
    }
}

__global__ void k_to_bf16(const float* __restrict__ x, int64_t n, bf16* __restrict__ y) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) y[i] = (bf16)x[i];
}

}  // namespace

struct pt_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    int members = 0, batch = 0;
    Layout L;
    int64_t t = 0;  // Adam steps taken
    float *params = nullptr, *grads = nullptr, *m1 = nullptr, *m2 = nullptr;
    bf16* wb = nullptr;
    float *X = nullptr, *Y = nullptr;
    int64_t n_data = 0;
    int32_t* order = nullptr;
    int64_t order_cap = 0;
    bf16* xb = nullptr;
    bf16* act[PT_MLP_LAYERS] = {};   // act[1..4]: hidden outputs
    float* slope[PT_MLP_LAYERS - 1] = {};  // gelu' of the hidden layers' pre-activations
    float* pred = nullptr;
    bf16* dz[PT_MLP_LAYERS] = {};  // gradients of the layers' outputs before GELU
    float* part = nullptr;         // squared errors per output tile
    float* colpart = nullptr;  // bias-gradient partial sums [layers][members][row chunks or tiles][kMaxWidth]
    float* loss = nullptr;
    int64_t loss_cap = 0;
    float* xin = nullptr;  // prediction inputs
    int64_t xin_cap = 0;
    // Prediction results on their way to the caller: pinned slots, each with
    // an event that marks its copy's end (the second slot and the events when a
    // result first needs them).
    float* slot[2] = {};
    int64_t slot_cap[2] = {};  // floats
    hipEvent_t slot_ev[2] = {};
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double last_ms = 0;
    // Training steps: [0] step index within the current call, [1] Adam steps
    // taken.  Up to eight steps are captured as a HIP graph per training call and
    // replayed (use_graphs), or enqueued kernel by kernel.
    int64_t* d_step = nullptr;
    float* bias_corr = nullptr;  // Adam's bias corrections of the step (finish_loss)
    bool use_graphs = true;
};

namespace {

int64_t act_z(const pt_mlp* m) { return (int64_t)m->batch * PT_MLP_HIDDEN; }
int64_t dz_z(const pt_mlp* m, int l) { return (int64_t)m->batch * kDims[l + 1]; }
int out_tiles(int rows) { return (rows + kColRows - 1) / kColRows * ((PT_MLP_OUT + kTile - 1) / kTile); }
int row_tiles(const pt_mlp* m) { return (m->batch + kTile - 1) / kTile; }
// Floats per layer slice of colpart: members x (row tiles) x kMaxWidth.
int64_t colpart_slice(const pt_mlp* m) { return (int64_t)m->members * row_tiles(m) * kMaxWidth; }

// Forward pass of every member on `rows` rows (at most batch) of b: outputs
// into pred, or (training) the loss and the output gradients.
void forward(pt_mlp* m, int rows, const Batch& b, bool training) {
    for (int l = 0; l < PT_MLP_LAYERS; ++l) {
        ForwardArgs g;
        memset(&g, 0, sizeof g);
        g.A = l == 0 ? nullptr : m->act[l];
        g.a_z = act_z(m);
        g.W = m->wb + m->L.w[l];
        g.bias = m->params + m->L.b[l];
        g.param_z = m->L.count;
        g.M = rows;
        g.N = kDims[l + 1];
        g.K = kDims[l];
        g.members = m->members;
        g.batch = b;
        const bool out = l == PT_MLP_LAYERS - 1;
        const int tiles = (g.N + kTile - 1) / kTile * ((rows + kTile - 1) / kTile) * m->members;
        if (!out) {
            if (training) g.out = m->slope[l];
            g.out_z = act_z(m);
            g.act = m->act[l + 1];
            g.act_z = act_z(m);
            if (l == 0 && training) g.xb = m->xb;
            (l == 0 ? k_forward<FWD_FIRST> : k_forward<FWD_HIDDEN>)<<<blocks_for_tiles(tiles), kGemmThreads, 0,
                                                                     m->stream>>>(g);
        } else if (!training) {
            g.out = m->pred;
            g.out_z = (int64_t)m->batch * PT_MLP_OUT;
            k_forward<FWD_OUT><<<blocks_for_tiles(tiles), kGemmThreads, 0, m->stream>>>(g);
        } else {
            g.act = m->dz[l];
            g.act_z = dz_z(m, l);
            g.part = m->part;
            g.colpart = m->colpart + l * colpart_slice(m);
            k_forward<FWD_LOSS><<<blocks_for_tiles(out_tiles(rows) * m->members), kGemmThreads, 0, m->stream>>>(g);
        }
    }
}

// Gradients of every member after forward(training), and the loss.  step (may
// be null): the training step counters.
void backward(pt_mlp* m, float* loss, int64_t loss_z, int64_t* step) {
    for (int l = PT_MLP_LAYERS - 1; l > 0; --l) {
        // dz_{l-1} = (dz_l W_l^T) * slope_{l-1}
        BackwardArgs g;
        memset(&g, 0, sizeof g);
        g.dz = m->dz[l];
        g.dz_z = dz_z(m, l);
        g.W = m->wb + m->L.w[l];
        g.param_z = m->L.count;
        g.M = m->batch;
        g.N = kDims[l];
        g.K = kDims[l + 1];
        g.members = m->members;
        g.slope = m->slope[l - 1];
        g.slope_z = act_z(m);
        g.out = m->dz[l - 1];
        g.out_z = dz_z(m, l - 1);
        g.colpart = m->colpart + (l - 1) * colpart_slice(m);
        g.finish = l == PT_MLP_LAYERS - 1;
        g.step = StepArgs{m->part, out_tiles(m->batch), m->members, (int64_t)m->batch * PT_MLP_OUT, loss, loss_z, step,
                          m->bias_corr};
        const int tiles = g.N / kTile * row_tiles(m) * m->members;
        k_backward<<<blocks_for_tiles(tiles) + g.finish, kGemmThreads, 0, m->stream>>>(g);
    }
}

// Weight and bias gradients after backward: Adam steps, or (adam false) left
// in grads.
void update(pt_mlp* m, bool adam, float lr) {
    UpdateArgs g;
    memset(&g, 0, sizeof g);
    for (int l = 0; l < PT_MLP_LAYERS; ++l) {
        g.act[l] = l == 0 ? m->xb : m->act[l];
        g.act_z[l] = l == 0 ? 0 : act_z(m);
        g.dz[l] = m->dz[l];
        g.dz_z[l] = dz_z(m, l);
        g.colpart[l] = m->colpart + l * colpart_slice(m);
    }
    g.R_hidden = row_tiles(m);
    g.R_out = (m->batch + kColRows - 1) / kColRows;
    g.members = m->members;
    g.batch = m->batch;
    g.count = m->L.count;
    g.grads = m->grads;
    g.p = m->params;
    g.m1 = m->m1;
    g.m2 = m->m2;
    g.pb = m->wb;
    g.lr = lr;
    g.bias_corr = m->bias_corr;
    const int blocks = blocks_for_tiles(member_tiles() * m->members) + kBiasBlocks * m->members;
    (adam ? k_update<true> : k_update<false>)<<<blocks, kGemmThreads, 0, m->stream>>>(g);
}

int upload_rows(pt_mlp* m, const int32_t* rows, int64_t n) {
    for (int64_t i = 0; i < n; ++i)
        if (rows[i] < 0 || rows[i] >= m->n_data) return fail(PT_EINVAL, "row %d outside the training set", rows[i]);
    if (n > m->order_cap) {
        dev_free(m->order);
        if (dev_alloc(&m->order, n)) return PT_ENOMEM;
        m->order_cap = n;
    }
    HIP_TRY(hipMemcpyAsync(m->order, rows, sizeof(int32_t) * n, hipMemcpyHostToDevice, m->stream));
    return PT_OK;
}

}  // namespace

extern "C" {

int64_t pt_mlp_param_count(void) { return Layout().count; }

int pt_mlp_create(int32_t members, int32_t batch, int32_t device, pt_mlp** out) {
    if (!out) return fail(PT_EINVAL, "null argument");
    *out = nullptr;
    if (members < 1 || members > 64) return fail(PT_EINVAL, "members %d outside [1, 64]", members);
    if (batch < 64 || batch % 64 || batch > 65536) return fail(PT_EINVAL, "batch %d: a multiple of 64 up to 65536", batch);
    HIP_TRY(hipSetDevice(device));
    pt_mlp* m = new pt_mlp();
    m->device = device;
    m->members = members;
    m->batch = batch;
    if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) {
        delete m;
        return fail(PT_EDEVICE, "hipStreamCreate failed");
    }
    const int64_t P = m->L.count * members;
    bool bad = dev_alloc(&m->params, P) || dev_alloc(&m->grads, P) || dev_alloc(&m->m1, P) || dev_alloc(&m->m2, P) ||
               dev_alloc(&m->wb, P) || dev_alloc(&m->xb, (int64_t)batch * PT_MLP_IN) ||
               dev_alloc(&m->pred, (int64_t)members * batch * PT_MLP_OUT) ||
               dev_alloc(&m->part, (int64_t)members * out_tiles(batch)) ||
               dev_alloc(&m->colpart, PT_MLP_LAYERS * colpart_slice(m)) || dev_alloc(&m->bias_corr, 2);
    for (int l = 1; l < PT_MLP_LAYERS && !bad; ++l) bad = dev_alloc(&m->act[l], members * act_z(m)) != 0;
    for (int l = 0; l < PT_MLP_LAYERS - 1 && !bad; ++l) bad = dev_alloc(&m->slope[l], members * act_z(m)) != 0;
    for (int l = 0; l < PT_MLP_LAYERS && !bad; ++l) bad = dev_alloc(&m->dz[l], members * dz_z(m, l)) != 0;
    if (bad) {
        const std::string msg = pt_last_error();
        pt_mlp_destroy(m);
        return fail(PT_ENOMEM, "%s", msg.c_str());
    }
    (void)hipEventCreate(&m->ev0);
    (void)hipEventCreate(&m->ev1);
    if (dev_alloc(&m->d_step, 2)) {
        pt_mlp_destroy(m);
        return PT_ENOMEM;
    }
    *out = m;
    return PT_OK;
}

int pt_mlp_set_params(pt_mlp* m, const float* params) {
    if (!m || !params) return fail(PT_EINVAL, "null argument");
    HIP_TRY(hipSetDevice(m->device));
    const int64_t P = m->L.count * m->members;
    HIP_TRY(hipMemcpyAsync(m->params, params, sizeof(float) * P, hipMemcpyHostToDevice, m->stream));
    HIP_TRY(hipMemsetAsync(m->m1, 0, sizeof(float) * P, m->stream));
    HIP_TRY(hipMemsetAsync(m->m2, 0, sizeof(float) * P, m->stream));
    k_to_bf16<<<grid_for(P, 256, 8192), 256, 0, m->stream>>>(m->params, P, m->wb);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(m->stream));
    m->t = 0;
    return PT_OK;
}

int pt_mlp_get_params(pt_mlp* m, float* params) {
    if (!m || !params) return fail(PT_EINVAL, "null argument");
    HIP_TRY(hipSetDevice(m->device));
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(hipMemcpy(params, m->params, sizeof(float) * m->L.count * m->members, hipMemcpyDeviceToHost));
    return PT_OK;
}

int pt_mlp_set_data(pt_mlp* m, const float* X, const float* Y, int64_t n) {
    if (!m || !X || !Y || n <= 0) return fail(PT_EINVAL, "bad training set");
    HIP_TRY(hipSetDevice(m->device));
    HIP_TRY(hipStreamSynchronize(m->stream));
    dev_free(m->X);
    dev_free(m->Y);
    if (dev_alloc(&m->X, n * PT_MLP_IN) || dev_alloc(&m->Y, n * PT_MLP_OUT)) return PT_ENOMEM;
    HIP_TRY(hipMemcpy(m->X, X, sizeof(float) * n * PT_MLP_IN, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(m->Y, Y, sizeof(float) * n * PT_MLP_OUT, hipMemcpyHostToDevice));
    m->n_data = n;
    return PT_OK;
}

int pt_mlp_train(pt_mlp* m, const int32_t* order, int32_t steps, float lr, float* loss_out) {
    if (!m || !order || steps < 1) return fail(PT_EINVAL, "bad arguments");
    if (m->n_data == 0) return fail(PT_ESTATE, "train before set_data");
    HIP_TRY(hipSetDevice(m->device));
    const int B = m->batch;
    if (int rc = upload_rows(m, order, (int64_t)steps * B)) return rc;
    if ((int64_t)steps * m->members > m->loss_cap) {
        dev_free(m->loss);
        if (dev_alloc(&m->loss, (int64_t)steps * m->members)) return PT_ENOMEM;
        m->loss_cap = (int64_t)steps * m->members;
    }
    // Every kernel of a step reads the step index and Adam count from
    // d_step, so one captured step serves all of them.
    const int64_t h_step[2] = {0, m->t};
    HIP_TRY(hipMemcpyAsync(m->d_step, h_step, sizeof h_step, hipMemcpyHostToDevice, m->stream));
    auto one_step = [&]() {
        forward(m, B, Batch{m->X, m->Y, m->order, m->d_step}, true);
        backward(m, m->loss, steps, m->d_step);
        update(m, true, lr);
    };
    // Steps per graph: 8 us pass between two graphs (100 steps of 5 x 1024, one
    // step per graph: 0.8 ms).
    const int per = std::min(steps, 8);
    // The instantiated graph, released on every return.
    struct ExecGuard {
        hipGraphExec_t e = nullptr;
        ~ExecGuard() {
            if (e) (void)hipGraphExecDestroy(e);
        }
    } exec;
    if (m->use_graphs) {
        hipGraph_t graph = nullptr;
        HIP_TRY(hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal));
        for (int k = 0; k < per; ++k) one_step();
        // Ends the capture whatever happened inside it; a failed launch
        // there is reported here.
        const hipError_t ce = hipStreamEndCapture(m->stream, &graph);
        if (ce != hipSuccess || !graph) {
            if (graph) (void)hipGraphDestroy(graph);
            return fail(PT_EDEVICE, "training graph capture: %s", hipGetErrorString(ce));
        }
        const hipError_t e = hipGraphInstantiate(&exec.e, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (e != hipSuccess) return fail(PT_EDEVICE, "training graph: %s", hipGetErrorString(e));
    }
    HIP_TRY(hipEventRecord(m->ev0, m->stream));
    for (int s = 0; s < steps;) {
        if (exec.e && s + per <= steps) {
            const hipError_t e = hipGraphLaunch(exec.e, m->stream);
            if (e != hipSuccess) return fail(PT_EDEVICE, "training graph launch: %s", hipGetErrorString(e));
            s += per;
        } else {
            one_step();
            ++s;
        }
    }
    m->t += steps;
    HIP_TRY(hipEventRecord(m->ev1, m->stream));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipEventSynchronize(m->ev1));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, m->ev0, m->ev1));
    m->last_ms = ms;
    if (loss_out) {
        std::vector<float> h((size_t)steps * m->members);
        HIP_TRY(hipMemcpy(h.data(), m->loss, sizeof(float) * h.size(), hipMemcpyDeviceToHost));
        // device layout [member][step] -> [step][member]
        for (int s = 0; s < steps; ++s)
            for (int k = 0; k < m->members; ++k) loss_out[(size_t)s * m->members + k] = h[(size_t)k * steps + s];
    }
    return PT_OK;
}

int pt_mlp_gradients(pt_mlp* m, const int32_t* rows, float* grads_out, float* loss_out) {
    if (!m || !rows || !grads_out || !loss_out) return fail(PT_EINVAL, "null argument");
    if (m->n_data == 0) return fail(PT_ESTATE, "gradients before set_data");
    HIP_TRY(hipSetDevice(m->device));
    const int B = m->batch;
    if (int rc = upload_rows(m, rows, B)) return rc;
    if (m->members > m->loss_cap) {
        dev_free(m->loss);
        if (dev_alloc(&m->loss, m->members)) return PT_ENOMEM;
        m->loss_cap = m->members;
    }
    forward(m, B, Batch{m->X, m->Y, m->order, nullptr}, true);
    backward(m, m->loss, 1, nullptr);
    update(m, false, 0.f);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(hipMemcpy(grads_out, m->grads, sizeof(float) * m->L.count * m->members, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(loss_out, m->loss, sizeof(float) * m->members, hipMemcpyDeviceToHost));
    return PT_OK;
}

int pt_mlp_predict(pt_mlp* m, const float* X, int64_t n, float* out) {
    if (!m || !X || !out || n < 0) return fail(PT_EINVAL, "bad arguments");
    HIP_TRY(hipSetDevice(m->device));
    if (n == 0) return PT_OK;
    if (n * PT_MLP_IN > m->xin_cap) {
        dev_free(m->xin);
        if (dev_alloc(&m->xin, n * PT_MLP_IN)) return PT_ENOMEM;
        m->xin_cap = n * PT_MLP_IN;
    }
    HIP_TRY(hipMemcpyAsync(m->xin, X, sizeof(float) * n * PT_MLP_IN, hipMemcpyHostToDevice, m->stream));
    const int B = m->batch;
    // Results go through two pinned slots, so that a part's way to the
    // caller's memory (a host copy, bound by its page faults) overlaps the
    // next parts' products and device copies: a part is one chunk of all
    // members, or rows of one member's chunk.  A result of one part takes one
    // slot and waits for the stream: nothing else to overlap, and a handle that
    // is asked once pays for one pinned allocation and no event (first call on
    // a new handle, 2 x 7: 123 us with both slots and events, 99 without; later
    // calls 60 and 54).
    const int64_t rows0 = std::min<int64_t>(B, n), all = m->members * rows0;
    const int64_t part_rows = std::min(rows0, kSlotRows);
    const bool whole = all <= kSlotRows, single = whole && n <= B;
    const int64_t want = (whole ? all : part_rows) * PT_MLP_OUT;
    for (int i = 0; i < (single ? 1 : 2); ++i) {
        if (want > m->slot_cap[i]) {
            m->slot_cap[i] = 0;
            HIP_TRY(hipStreamSynchronize(m->stream));
            if (m->slot[i]) HIP_TRY(hipHostFree(m->slot[i]));
            m->slot[i] = nullptr;
            if (hipHostMalloc((void**)&m->slot[i], sizeof(float) * want) != hipSuccess)
                return fail(PT_ENOMEM, "hipHostMalloc of %lld bytes failed", (long long)(sizeof(float) * want));
            m->slot_cap[i] = want;
        }
        if (!single && !m->slot_ev[i]) HIP_TRY(hipEventCreateWithFlags(&m->slot_ev[i], hipEventDisableTiming));
    }
    struct Part {
        int64_t at = 0;             // first row of the result
        int rows = 0, members = 0;  // members of consecutive blocks of n rows
    } pending[2];
    int next = 0;
    auto drain = [&](int i) -> int {
        Part& q = pending[i];
        if (q.rows == 0) return PT_OK;
        HIP_TRY(single ? hipStreamSynchronize(m->stream) : hipEventSynchronize(m->slot_ev[i]));
        const size_t len = (size_t)q.rows * PT_MLP_OUT;
        for (int k = 0; k < q.members; ++k)
            memcpy(out + (size_t)(q.at + k * n) * PT_MLP_OUT, m->slot[i] + k * len, sizeof(float) * len);
        q.rows = 0;
        return PT_OK;
    };
    int rc = PT_OK;
    for (int64_t i0 = 0; i0 < n && !rc; i0 += B) {
        const int rows = (int)std::min<int64_t>(B, n - i0);
        forward(m, rows, Batch{m->xin + i0 * PT_MLP_IN, nullptr, nullptr, nullptr}, false);
        HIP_TRY(hipGetLastError());
        for (int k = 0; k < m->members && !rc; k += whole ? m->members : 1)
            for (int r0 = 0; r0 < rows && !rc; r0 += (int)part_rows) {
                const int i = next, count = std::min(rows - r0, (int)part_rows);
                if ((rc = drain(i))) break;
                const size_t len = sizeof(float) * count * PT_MLP_OUT;
                HIP_TRY(hipMemcpy2DAsync(m->slot[i], len, m->pred + ((int64_t)k * B + r0) * PT_MLP_OUT,
                                         sizeof(float) * B * PT_MLP_OUT, len, whole ? m->members : 1,
                                         hipMemcpyDeviceToHost, m->stream));
                if (!single) HIP_TRY(hipEventRecord(m->slot_ev[i], m->stream));
                pending[i] = Part{k * n + i0 + r0, count, whole ? m->members : 1};
                next = 1 - next;
            }
    }
    for (int i = 0; i < 2 && !rc; ++i) rc = drain((next + i) & 1);
    return rc;
}

int pt_mlp_use_graphs(pt_mlp* m, int32_t on) {
    if (!m) return fail(PT_EINVAL, "null handle");
    m->use_graphs = on != 0;
    return PT_OK;
}

double pt_mlp_last_train_ms(pt_mlp* m) { return m ? m->last_ms : -1.0; }

void pt_mlp_destroy(pt_mlp* m) {
    if (!m) return;
    (void)hipSetDevice(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    dev_free(m->params);
    dev_free(m->grads);
    dev_free(m->m1);
    dev_free(m->m2);
    dev_free(m->wb);
    dev_free(m->X);
    dev_free(m->Y);
    dev_free(m->order);
    dev_free(m->xb);
    for (int l = 1; l < PT_MLP_LAYERS; ++l) dev_free(m->act[l]);
    for (int l = 0; l < PT_MLP_LAYERS - 1; ++l) dev_free(m->slope[l]);
    for (int l = 0; l < PT_MLP_LAYERS; ++l) dev_free(m->dz[l]);
    dev_free(m->bias_corr);
    dev_free(m->pred);
    dev_free(m->part);
    dev_free(m->colpart);
    dev_free(m->loss);
    dev_free(m->xin);
    for (int i = 0; i < 2; ++i) {
        if (m->slot[i]) (void)hipHostFree(m->slot[i]);
        if (m->slot_ev[i]) (void)hipEventDestroy(m->slot_ev[i]);
    }
    if (m->ev0) (void)hipEventDestroy(m->ev0);
    if (m->ev1) (void)hipEventDestroy(m->ev1);
    dev_free(m->d_step);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

}  // extern "C"
