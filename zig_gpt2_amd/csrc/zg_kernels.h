// zg_kernels.h — host-callable launchers of the HIP kernels (internal to libzgpt2_hip).
#pragma once
#include "zg_common.h"

namespace zg {

// Device-side decode control block (lives in the model arena; read by kernels so that one
// captured hipGraph replays for every position).
struct StepCtrl {
    int step;      // 0-based decode step s; sequence length T = s + 1 while a step runs
    int seq_len;   // T of the step in flight (written by the embed kernel)
    int mode;      // 0: generate loop (tokens from prompts / previous argmax), 1: forced tokens
    int n_partials;  // number of lm_head argmax partials per sequence (grid of the lm_head GEMV)
};

// ------------------------------------------------------------------------------------ GEMV
enum GemvPrologue { PRO_NONE = 0, PRO_LAYERNORM = 1, PRO_ATTN_MERGE = 2 };
enum GemvEpilogue { EPI_STORE = 0, EPI_RESIDUAL = 1, EPI_GELU = 2, EPI_QKV = 3, EPI_ARGMAX = 4 };
enum WeightType { WT_BF16 = 0, WT_F32 = 1 };

constexpr int kAttnChunk = 256;       // KV positions per attention workgroup (4 waves x 64)
constexpr int kPartStride = 64 + 2;   // floats per attention partial: o[hd<=64], m, l

struct GemvArgs {
    // y[m][n] = epilogue( sum_k prologue(x)[m][k] * W[n][k] + bias[n] ),  m < M, n < N
    const void* W;  // [N][K], bf16 bits or fp32, K contiguous (ops.Linear.weight layout)
    const float* bias;  // [N] or nullptr
    int N, K, M;
    int rows_per_wave;
    int waves_per_wg;  // filled by gemv_plan (M == 1 kernels may run as 1..4-wave workgroups)
    int prologue, epilogue;
    // PRO_NONE / PRO_LAYERNORM input
    const float* x;  // [M][x_stride]
    int x_stride;
    const float* ln_g;
    const float* ln_b;
    float eps;
    // PRO_LAYERNORM, M == 1: the LayerNorm folded out of the dot product (launch_ln_fold): c2[n] = sum_k W g,
    // c3[n] = sum_k W b + bias[n]; null = use the kernel that normalises the input first
    const float* ln_c2;
    const float* ln_c3;
    // PRO_ATTN_MERGE input: partials [M][H][max_splits][kPartStride]
    const float* part;
    int n_heads, head_dim, max_splits;
    const StepCtrl* ctrl;  // seq_len for the merge / KV scatter position
    int t_hi;  // launch-time upper bound of seq_len (same 256-position chunk as seq_len); 0 = read ctrl
    // EPI_STORE / EPI_RESIDUAL / EPI_GELU
    float* y;
    int y_stride;
    const float* resid;  // may alias y
    int resid_stride;
    // EPI_QKV: q [M][E]; caches [M][H][ctx][hd]
    float* q;
    void* k_cache;
    void* v_cache;
    int ctx;
    int kv_mode;   // 0 fp32, 1 fp16, 2 B24 (bf16 plane + byte plane `kv_lo` bytes further on)
    size_t kv_lo;
    // EPI_ARGMAX: optional logits [M][logits_stride]; partials [M][gridDim.x]
    float* logits;
    int logits_stride;
    float* part_val;
    int* part_idx;
    // split-K over workgroups (batched wide Linears): combine workspace [sk_tiles][4][128] floats and FOUR counters per
    // tile (zero between launches: the last arriver resets its counter; the 16-wave kernel uses counter [tile], the
    // four-wave plane-fed kernel one per wave, [4 tile + wave]); kslices is filled by gemv_plan
    float* sk_ws;
    int* sk_cnt;
    int sk_tiles;
    int kslices;
    // lock-step batch on the matrix cores: activation planes in global memory (zg_common.h plane_elem).  pl_in: the
    // input rows arrive as planes written by the previous kernel (PRO_LAYERNORM: planes of g * x, x itself is read for
    // the row statistics only; PRO_NONE: planes of x).  pl_out: this kernel's output rows (after residual / GELU) are
    // also written as planes, scaled by pl_g[n] when given (the next LayerNorm's gain); EPI_GELU with y == nullptr
    // writes only the planes.
    const bf16_t* pl_in;
    bf16_t* pl_out;
    const float* pl_g;
    // K slices of the four-wave plane-fed kernel meet by TAGGED DATA instead of tickets: slices 1.. store (value, tag) as one
    // 8-byte word, slice 0 polls until the tags are this launch's — one memory-side round trip instead of three.
    // tag = *epoch << 8 | launch_id: epoch is advanced by the embed kernel at every step, launch_id (1..255) is unique
    // among the launches of a step that share sk_tag [sk_tiles][4][128].
    const unsigned* epoch;
    unsigned launch_id;
    unsigned long long* sk_tag;
    unsigned* fault;  // set to 1 by a poller whose bounded wait ran out (the host fails the call loudly: api_gpt.hip check_fault)
    unsigned spin_limit;  // polls before a poller gives up (2^20; ZGPT2_TAG_SPIN_LIMIT for the test of the failure path)
    // LayerNorm statistics by tile: a producer of x (four-wave plane-fed kernel, embed kernel) also writes, per 16-column tile
    // and batch row, the sum and the sum of squares of its 16 outputs, st_out [8][N / 16][2]; the LayerNorm-fed consumer
    // adds the tiles (st_in) instead of reading x again — a third of its vector-memory traffic
    float* st_out;
    const float* st_in;
    const float* zero;        // device pointer to a few zero floats (stand-in for absent bias / residual)
    unsigned long long* dbg;  // diagnostic timestamps (only read by -DZG_STAMPS builds)
    unsigned* progress;       // launch counter followed by the side-stream prefetcher (prefetch.hip); null = not counted
};

// Whether launch_gemv can run this M x K at all (batched kernels keep the M input rows in LDS).
bool gemv_supported(const GemvArgs& a, int weight_type);
// Whether this launch may take its input rows as planes in global memory (GemvArgs.pl_in).
bool gemv_planes_ok(const GemvArgs& a, int weight_type);
// ... and whether it can write its output rows as planes (GemvArgs.pl_out).
bool gemv_planes_producer_ok(const GemvArgs& a, int weight_type);
// Whether a planned plane-fed launch runs as the four-wave kernel (the one that writes / reads the tile statistics).
bool gemv_pl4_ok(const GemvArgs& a, int weight_type);
// Fills rows_per_wave and returns the grid size for the given problem.
int gemv_plan(GemvArgs& a, int weight_type = WT_F32);
int gemv_kslices(const GemvArgs& a);
// Rows of W that one workgroup of the planned launch reads (block b: rows b * r .. (b + 1) * r - 1); 0 = another mapping
int gemv_rows_per_wg(const GemvArgs& a, int weight_type);
int launch_ln_fold(const void* W, int weight_type, const float* g, const float* b, const float* bias, int N, int K, float* c2,
                   float* c3, hipStream_t s);
int launch_gemv(const GemvArgs& a, int weight_type, int grid, hipStream_t s);

// ------------------------------------------------------------------------------------ attention
struct AttnArgs {
    const float* q;  // [B][H*hd]
    const void* k;   // element (b,h,t,d) at b*stride_b + h*stride_h + t*stride_t + d
    const void* v;
    long stride_b, stride_h, stride_t;
    int kv_mode;   // 0 fp32, 1 fp16, 2 B24: bf16 plane at k / v, byte plane (same element strides) kv_lo bytes further on
    size_t kv_lo;
    int n_heads, head_dim, batch;
    const StepCtrl* ctrl;  // seq_len read from ctrl->seq_len when non-null
    int seq_len;           // used when ctrl == nullptr
    int t_hi;              // launch-time upper bound of seq_len in the same 64-position bucket (>= seq_len)
    int max_splits;
    float* part;  // [B][H][max_splits][kPartStride]
    unsigned* progress;  // see GemvArgs
    // lock-step batch with activation planes: the last split of (b, h) to arrive merges them and writes the head's output as
    // planes [3][8][H * 64] (plane_elem) for the c_proj Linear; merge_cnt = one zeroed counter per (b, h)
    bf16_t* pl_out;
    int* merge_cnt;
    // ... or, with part_tag [B][H][max_splits][66] given, split 0 merges: the other splits store (value, tag) words and
    // split 0 polls them (see GemvArgs.sk_tag for the tag)
    const unsigned* epoch;
    unsigned launch_id;
    unsigned long long* part_tag;
    unsigned* fault;  // see GemvArgs.fault
    unsigned spin_limit;
};
int launch_attn_decode(const AttnArgs& a, hipStream_t s);
// the op tier's general path for head_dim != 64 (fp32, one workgroup per (sequence, head))
int launch_attn_any_dim(const float* q, const float* k, const float* v, long stride_b, long stride_h, long stride_t, int batch, int n_heads,
                        int head_dim, int seq_len, float* out, hipStream_t s);
// Standalone merge (op tier): out[b][h*hd+d] = sum_s w_s o_s / sum_s w_s l_s
int launch_attn_merge(const float* part, int batch, int n_heads, int head_dim, int max_splits,
                      int seq_len, float* out, hipStream_t s);

// ------------------------------------------------------------------------------------ elementwise
int launch_epoch_bump(unsigned* epoch, hipStream_t s);  // measurement chains: advance the tag epoch (api_gpt.hip zg_gpt_time_kernel)
int launch_layernorm(float* x, int rows, int n, const float* g, const float* b, float eps, hipStream_t s, unsigned* done_flag = nullptr,
                     unsigned done_seq = 0, bool* announced = nullptr, float* shadow = nullptr);
int launch_gelu(float* x, size_t n, hipStream_t s, unsigned* done_flag = nullptr, unsigned done_seq = 0, bool* announced = nullptr, float* shadow = nullptr);
int launch_softmax(float* x, size_t n, hipStream_t s, unsigned* done_flag = nullptr, unsigned done_seq = 0, bool* announced = nullptr);
int launch_done_flag(unsigned* flag, unsigned seq, hipStream_t s);
struct CopySegs {  // up to four device -> pinned-host segments (16-byte aligned, multiples of 4 bytes)
    const void* src[4];
    void* dst[4];
    unsigned bytes[4];
    int n;
};
int launch_copy_out_done(const CopySegs& segs, unsigned* flag, unsigned seq, hipStream_t s);
int launch_copy2_f32(const float* a, float* da, const float* b, float* db, size_t n, hipStream_t s);
int launch_embedding(const float* w, size_t emb_dim, const size_t* idx, size_t n_idx, size_t n_rows,
                     float* out, int* d_oob_flag, hipStream_t s, unsigned* done_flag = nullptr, unsigned done_seq = 0, bool* announced = nullptr);
int launch_split_qkv(const float* in, size_t rows, size_t n_embed, size_t split_idx, float* out, hipStream_t s);
int launch_transpose(const float* in, size_t batch, size_t t, size_t n, size_t h, float* out, hipStream_t s);
int launch_copy_f32(const float* in, float* out, size_t n, hipStream_t s);
int launch_f32_to_bf16(const float* in, bf16_t* out, size_t n, hipStream_t s);
// fp32 [rows][K] -> bf16 [rows][3K] = [hi | mid | lo], hi + mid + lo == x exactly
int launch_split3(const float* in, size_t rows, int K, bf16_t* out, hipStream_t s);
// fp32 [rows][K] of one or two matrices (the second may have none) -> fp16 [rows][2K] = [hi | lo] of the rows times 2^-exps[row], which brings their
// largest value to [2^14, 2^15): elementwise.hip
// In front of a Linear's products from kSplit2MinK columns on: shorter sums of three exact bf16 terms are closer to 64 bits than two fp16 terms can be
// (4096 rows, 3072 outputs: 512 columns 1.27e-7 against 1.34e-7, 576 1.35e-7 and 1.39e-7, 640 1.43e-7 both, 704 1.51e-7 and 1.48e-7, 768 1.58e-7 and 1.52e-7, 1536 2.32e-7 and
// 1.96e-7; us a call 90 : 66, 95 : 69, 103 : 72, 109 : 76, 117 : 81, 207 : 136).
constexpr size_t kSplit2MinK = 640;
// A prompt Linear's sums are in units of 2^(a + e), a the exponent of the activations and e of the weight's row: a row's exponent is never so low that its bias leaves
// fp32's range in those units (where the persistent GEMM starts its sums) or the unit itself does.  What such a row of tiny weights loses lies some 60 binades
// below the bias, or beyond the smallest fp32 number.
struct PlaneFloor {
    const int* a = nullptr;
    const float* bias = nullptr;
};
// What the pass over both operands of a Linear saw of their rows.  A value below 2^-17 of its row's largest loses bits in two fp16 terms: 2^-39 of the largest is what is
// left out.  In a sum of products that is nothing as long as they are few and there are others beside them: three quarters of one operand's row and three
// eighths of the other's within 2^-10 of their largest value leave an eighth of the products above 2^-20 of the two largest, and what a 64th of the values
// in either row loses is below 2^-21 of the sum of |x w|.  Rows of normal values, of ReLU or GELU outputs, rows with a value some hundred times the others' are so; a
// row with one of a million, or of softmax weights, need not be.  Outputs of rows that are not are worked out again: as plain sums where the rows are few, else the kernels
// leave at once and the call takes exact planes.
// Words are equal to the call's number where the thing is so; rows are counted by how many of their sixteen words are.
enum { SEEN_ANY = 0 /* a row that is not even */, SEEN_ODD = 1 /* one with a value that is not finite */, SEEN_ROWS = 16, SEEN_X_UNEVEN = 0, SEEN_X_SPARSE = 1, SEEN_W_UNEVEN = 2,
       SEEN_W_SPARSE = 3, kSeenWords = SEEN_ROWS + 4 * 16, kSeenFew = 12 };
enum { MARK_ODD = 1, MARK_UNEVEN = 2 /* fewer than three quarters */, MARK_SPARSE = 4 /* than three eighths, or too many small ones */ };
struct SplitSeen {
    unsigned* words = nullptr;
    unsigned* host = nullptr;  // pinned: [0] the call was refused, [1] it has rows to be worked out again, [2] rows with values that are not finite
    int* marks = nullptr;      // of x's rows, then w's (in whole fours)
    unsigned call = 0;
};
struct Split2Job {
    const float* in;
    uint16_t* out;
    int* exps;
    int rows;
    size_t lo = 0;           // the second plane lies this many elements behind the first (0: beside it, rows of 2K)
    float* norms = nullptr;  // 2-norms of the rows
    const int* one = nullptr;  // the exponent of every row; else each gets its own, ...
    PlaneFloor floor;          // ... no lower than this
    uint16_t* rest = nullptr;  // what two terms leave (the 24th bit of one value in four), a plane of its own
};
// for the test hooks of one Linear and one attention: rows of three bf16 planes -> fp32, rows of two fp16 planes times 2^exp -> three bf16 planes
int launch_join_planes(const uint16_t* in, const int* exp, int rows, int K, int planes, float* out, hipStream_t s);
int launch_join_planes(const uint16_t* in, const int* exp, int rows, int K, int planes, bf16_t* out, hipStream_t s);
// bf16 [rows][K] -> one plane of fp16 (a bf16 value has 8 significant bits: exact down to 2^-32 of its row's largest)
int launch_plane_bf16(const bf16_t* in, int rows, int K, uint16_t* out, int* exps, float* norms, hipStream_t s, const PlaneFloor& floor = PlaneFloor{});
int launch_split2(const Split2Job& a, const Split2Job& b, int K, hipStream_t s, const SplitSeen& seen = SplitSeen{});
// rows [from_row, ctx) of every (cache, sequence x head) strip set to zero: n_caches caches cache_stride bytes apart, each holding a
// plane of [strips][ctx] rows of row_bytes at plane_off (api_gpt.hip clear_kv: what a new sequence must not inherit)
int launch_kv_clear_tail(void* base, int n_caches, size_t cache_stride, size_t plane_off, int row_bytes, int strips, int ctx, int from_row,
                         hipStream_t s);

// ------------------------------------------------------------------------------------ MFMA GEMM
// C[M,N] = A[M,K] * B[N,K]^T (+ bias) (optional GELU); bf16 operands, fp32 accumulate; C bf16 or fp32.
int launch_gemm_bf16_nt(const bf16_t* A, const bf16_t* B, const float* bias, void* C, int M, int N, int K, int ldc,
                        bool gelu, bool out_bf16, hipStream_t s);
// The same kernel over a list of (A plane, B plane) pairs: A is [M][lda] holding planes of K = 64 kpp columns each
// (plane p at column p K), B is [N][ldb] likewise; C = sum over pairs of A_plane[pa] * B_plane[pb]^T (+ bias).
// fp32 operands split exactly into bf16 hi + mid + lo planes make the bf16 matrix cores deliver fp32-grade
// products (every bf16 x bf16 product is exact in fp32): planes {(2,0),(1,0),(0,0)} for exact-bf16 weights,
// six pairs for arbitrary fp32 weights.  Pair i's planes sit in bits [4i, 4i + 4) of pa_bits / pb_bits.
struct GemmPlanes {
    int lda, ldb;  // row lengths in elements
    int kpp;       // K-steps (of 64) per plane
    int npairs;
    unsigned pa_bits, pb_bits;
    bool b_plane_major;  // B's planes are whole [N][ldb] matrices one behind the other (the model's fp32-weight planes), not column blocks of a row
};
int launch_gemm_planes(const bf16_t* A, const bf16_t* B, const float* bias, void* C, int M, int N, const GemmPlanes& pl,
                       int ldc, bool gelu, bool out_bf16, hipStream_t s);
int launch_gemm_s4(const bf16_t* A, const bf16_t* B, const float* bias, void* C, int M, int N, const GemmPlanes& pl, int ldc,
                   bool gelu, bool out_bf16, int bn, hipStream_t s);  // gemm_s4.hip
bool gemm_s4_args_ok(const GemmPlanes& pl, int ldc);            // the bounds of gemm_s4_kernel's packed arguments
// ... with planes of fp16 (launch_split2): what the sums of output row m and column n are multiplied with, 2^(a[m] + w[n]) (a_each; else a[0] for every row)
struct PlaneExps {
    const int* a;
    const int* w;
    bool a_each;
};
int launch_gemm_s4_f16(const uint16_t* A, const uint16_t* B, const float* bias, float* C, int M, int N, const GemmPlanes& pl, int ldc, const PlaneExps& ex, const SplitSeen& seen,
                       hipStream_t s);  // (nothing is computed of a call that is refused: SplitSeen)
// ... and its epilogue kinds for the whole-prompt Linears (gemm_s4.hip; PrefillQkv below)
enum { S4_PLAIN = 0, S4_PARTIAL = 1, S4_QKV = 2, S4_SPLIT2 = 3, S4_RELU2 = 4 };
int launch_gemm_s4_relu2(const bf16_t* A, const bf16_t* B, const float* bias, void* C, int M, int N, const GemmPlanes& pl, int ldc, bool out_bf16, hipStream_t s);
struct PrefillQkv;
struct PrefillA;
struct PrefillW;
struct PlaneOut;
int launch_gemm_s4_prefill(const PrefillA& A, const PrefillW& W, const float* bias, void* C, int M, int N, int K, int kind, int n_slices,
                           const PrefillQkv* qkv, const PlaneOut& po, hipStream_t s);
int gemm_s4_stamps(unsigned long long* out, size_t n_words);  // diagnostic (ZGPT2_GEMM_DBG bit 256)
int gemm_s4_fault(unsigned* out);  // 1: a stream-K consumer of gemm_s4 gave up waiting for its producer since the last call (results wrong)
int gemm_debug_stamps(unsigned long long* out, size_t n_words);  // of the kernel generation launched last
unsigned long long gemm_mfma_launch_count();  // launches of the persistent MFMA GEMMs so far (tests assert the path taken)
void gemm_note_launch();
// fp32 Linears X [M][K], W [N][K] of few rows and of a medium number of rows (linear_tiles.hip).  Two to fifteen rows: K a multiple of 8.
bool linear_few_ok(size_t M, size_t N, size_t K);
unsigned long long linear_few_mfma_launch_count();  // launches of linear_few_mfma_kernel so far
int launch_linear_few(const float* X, const float* W, const float* bias, float* Y, int M, int N, int K, hipStream_t s);
// Nine rows and more: K a multiple of 64; slabs: linear_tiles_slices(M, N, K) * M * N floats where that is more than one slice.
bool linear_tiles_pay(size_t M, size_t N, size_t K, bool planes);  // planes: beside the persistent GEMM on fp16 planes where it takes them; else on exact bf16 ones
double linear_tiles_us(size_t M, size_t N, size_t K);  // what a call by it takes, in us
double linear_split_mb(size_t M, size_t N, size_t K), linear_split_us(size_t M, size_t N, size_t K);  // the pass in front of the kernels on planes of two terms
// Outputs of rows (of X and W) that are not for two terms or have values that are not finite, as plain fp32 sums
int launch_linear_marked_rows(const float* X, const float* W, const float* bias, float* Y, int M, int N, int K, const SplitSeen& seen, hipStream_t s);
int linear_tiles_slices(size_t M, size_t N, size_t K);
int launch_linear_tiles(const float* X, const float* W, const float* bias, float* Y, int M, int N, int K, float* slabs, hipStream_t s);

// ------------------------------------------------------------------------------------ prefill (prefill.hip)
// Whole-prompt forward.  Activations feeding a GEMM are two-term fp16 planes (zg_common.h split2_f16), [M][kPair * K] = [hi | lo] of the
// fp32 values times 2^-exp, exp one number for all of them: a bound on the values that holds for any input follows from the weights alone
// (launch_prefill_bounds), so that it is known before they are.
constexpr int kPair = 2;
struct PlaneOut {
    const int* exp;
    int coarse;  // ZG_GPT_PREFILL_2PLANE: values rounded to 16 significant bits first
};
// a Linear's weight: fp16 planes [planes][N][K] of its rows times 2^-exps[row]; one plane holds a bf16 value, two 23 bits of an fp32 value, and the third behind them, where
// there is one (models of fewer than kNearColumns columns), the last
struct PrefillW {
    const uint16_t* p;
    const int* exps;
    int planes;
    bool rest = false;
};
constexpr size_t kNearColumns = 512;
enum PrefillEpilogue { PF_F32 = 0, PF_RESID = 1, PF_GELU_SPLIT = 2, PF_PARTIAL = 3 /* internal: split-K slice */, PF_QKV = 4, PF_LINEAR = 5, PF_LINEAR_PART = 6 /* internal: Linear.forward, and a slice of one */ };
int launch_embed_prefill(const int* tokens, int token_stride, int B, int P, const void* wte, const void* wpe,
                         int weight_type, int E, float* x, hipStream_t s);
int launch_ln_split(const float* x, int M, int E, const float* g, const float* b, float eps, uint16_t* out, const PlaneOut& po, hipStream_t s);
// C = A[M][K] * W[N][K]^T + bias; PF_F32: fp32 C[M][ldc]; PF_RESID: C += ...; PF_GELU_SPLIT: planes C[M][kPair N] of gelu(...), as po says
// ws: fp32 workspace for split-K partial sums (used when the output has too few tiles to fill the chip).
// ln (PF_RESID only, may be null): LayerNorm of the updated rows, written as split planes to ln->out — fused
// into the split-K tail when there is one, a separate launch_ln_split otherwise.
// PF_QKV: fp32 store of the qkv rows (row m = b P + t) AND the cache append of ops.zig:152-157 for the K / V
// columns, into the head-major caches [b][h][ctx][64] (fp32 or fp16).
struct PrefillQkv {
    int P, E, H, ctx, kv_mode;
    void* k_cache;
    void* v_cache;
    size_t kv_lo;  // kv_mode 2: byte offset of the low-mantissa plane
    // stream-K hand-over of the persistent GEMM (gemm_s4.hip, S4_QKV with 1.5 rounds of tiles): workspace for the producers'
    // accumulators (196608 B per shared tile), one flag word per (shared tile, wave), the launch's epoch (flags of earlier
    // launches are smaller); null = whole tiles only
    void* sk_ws = nullptr;
    size_t sk_ws_bytes = 0;
    unsigned* sk_flags = nullptr;
    unsigned sk_flags_words = 0;  // words behind sk_flags (4 per shared tile: G / 2 tiles for G workgroups)
    unsigned sk_epoch = 0;
};
struct PrefillLn {
    const float* g;
    const float* b;
    float eps;
    uint16_t* out;
    PlaneOut po;
};
// a: the exponents of A's rows (each: one for every row, else one for all)
struct PrefillA {
    const uint16_t* p;
    const int* exp;
    bool each;
};
int launch_prefill_gemm(const PrefillA& A, const PrefillW& W, const float* bias, void* C, int M, int N, int K, int ldc, int epi,
                        float* ws, size_t ws_floats, const PrefillLn* ln, hipStream_t s, const PrefillQkv* qkv = nullptr, const PlaneOut& po = PlaneOut{});
// prefill_ring.hip: whole-prompt Linears of some hundred rows.  The route: K slices (slabs of a residual Linear, else 1), 0 = not taken; tm: rows / 64 of a tile.
int prefill_ring_route(int M, int N, int K, bool resid, bool planes, size_t ws_floats, bool force, int* tm);
int launch_prefill_ring(const PrefillA& A, const PrefillW& W, const float* bias, void* C, int M, int N, int K, int ldc, int epi, int tm, int n_sp, const PrefillQkv& qa,
                        const PlaneOut& po, hipStream_t s);
// The exponents of a layer's activations, from its weights: of a normed x g + b, with x's rows no longer than sqrt(E), column e is no larger than sqrt(E) |g_e| + |b_e|, and
// an output of a Linear behind it no larger than sqrt(E) |g w| + |w b + bias| (2-norm over the row's columns; launch_row_bounds).  Bounds that hold for
// any input, and no looser than they have to be: a trained layer's gains and rows differ by factors of ten and more, and what lies far below its bound has
// fewer bits (2^-17 of the bound and more: all of two terms; below, 2^-40 of the bound is left out).  exps: kBounds of them (enum).
enum { PB_LN1 = 0, PB_Q = 1, PB_K = 2, PB_V = 3, PB_LN2 = 4, PB_GELU = 5, kBounds = 8 };
struct PrefillBounds {
    const float *ln_1_g, *ln_1_b, *ln_2_g, *ln_2_b;
    const double *c_attn_rows, *c_fc_rows;  // bounds on the outputs (launch_row_bounds)
    int* exps;
};
int launch_row_bounds(const void* W, int weight_type, const float* g, const float* b, const float* bias, int rows, int E, double* out, hipStream_t s);
int launch_prefill_bounds(const PrefillBounds& b, int E, hipStream_t s);
// ... and the fp32 Linears of the op tier with some hundred rows on the same kernel, behind a pass that splits both operands.  The route: slices of K (0: not taken), tm
// as above; scratch: linear_ring_scratch bytes.
int linear_ring_route(size_t M, size_t N, size_t K, int* tm);
unsigned long long linear_ring_launch_count();  // Linears it has taken so far
size_t linear_ring_scratch(size_t M, size_t N, size_t K, int n_sp);
int launch_linear_ring(const float* X, const float* W, const float* bias, float* Y, int M, int N, int K, int tm, int n_sp, char* scratch, SplitSeen* seen, hipStream_t s);  // (seen->marks: set)
bool prefill_rows_wide(int M, int N, int planes);  // the 128-row kernels' tiles: 256 columns for 128
void prefill_force_route(int kernel, int slices);  // zg_debug_prefill_route / _linear: pin the GEMM family (1 gemm_s4, 2 the 128-row kernels, 3 prefill_ring) and the K slices
// out[M][kPair E] = planes of the causal attention of the q / k / v columns of qkv[M][3E], M = B P rows ordered (b, t)
// (attn_prefill.hip: matrix cores on two-term fp16 planes).  exps: kBounds of them; the output has v's (a weighted mean of rows of v is no larger than they are).
int launch_attn_prefill(const float* qkv, uint16_t* out, int B, int P, int E, int H, const float* k_cache_or_null, const float* v_cache_or_null, int ctx, const int* exps,
                        int coarse, hipStream_t s, bool by_groups = false, unsigned long long* stamps = nullptr);

// GPT.sample tail: in-place softmax(logits / temp) per sequence + inverse-CDF draw with uniform u[b].
// part_val / n_part / part_stride: the per-workgroup maxima lm_head's argmax epilogue left (the row maximum without a pass over the
// logits); seg_ws: sample_workspace_floats(batch) floats; write_probs: leave softmax(logits / temp) in the logits rows
int launch_sample(float* logits, int batch, int vocab, float temp, const float* u, const float* part_val, int n_part, int part_stride, float* seg_ws,
                  int* token_out, bool write_probs, hipStream_t s);
size_t sample_workspace_floats(int batch);

// Decode-step head kernel: token selection (+ argmax finalisation of the previous step) and
// x = wte[token] + wpe[pos].
struct EmbedArgs {
    // the first 14 dwords are preloaded into SGPRs (zg_common.h ZG_PIN): what the first loads of the kernel depend on
    StepCtrl* ctrl;
    const float* part_val;   // [B][n_partials]
    const int* part_idx;
    int part_stride;
    int n_partials;          // lm_head grid size
    const int* prompt;       // [B][prompt_stride]
    const int* prompt_len;   // [B]
    int batch;
    int prompt_stride;
    // ... the rest is fetched from the kernarg segment under those loads
    const int* forced;       // [B] (mode 1)
    const void* wte;  // [V][E] bf16 or fp32
    const void* wpe;  // [ctx][E]
    int weight_type;
    int n_embed, vocab;
    int* cur_token;          // [B]
    int* out_tokens;         // [B][out_stride]
    int out_stride;
    float* x;                // [B][E]
    bf16_t* pl_out;          // optional planes of pl_g * x for the first Linear of the lock-step batch (GemvArgs.pl_in)
    const float* pl_g;
    unsigned* epoch;         // optional step counter behind the tagged hand-overs (GemvArgs.sk_tag): +1 when a step starts
    float* st_out;           // optional LayerNorm statistics by tile of x (GemvArgs.st_in): [8][n_embed / 16][2]
    int finish_only;         // 1: only record the greedy pick of the last step; 2: argmax -> cur_token
    unsigned* progress;      // set to (T << 8) | 1 (and the XCD of this block beside it) when a step starts; the other decode kernels add 1 each
    const int* sampled;      // [B] (mode 2: generate with the sampler) the token sample_step_kernel drew from the previous step's logits
};
int launch_embed_step(const EmbedArgs& a, hipStream_t s);
// GPT.sample's tail (src/main.zig:200-206) inside the generate loop: temperature and seed live in device memory (one captured
// graph serves every call), the uniform of (sequence b, position T) is the library's counter PRNG of (seed, T, b) — what
// zg_gpt_sample uses when it is given no uniforms
struct SampleParams {
    float inv_temp;
    unsigned pad;
    unsigned long long seed;
};
int launch_sample_step(float* logits, int batch, int vocab, const SampleParams* params, const StepCtrl* ctrl, const float* part_val, int n_part,
                       int part_stride, float* seg_ws, int* token_out, hipStream_t s);

// ------------------------------------------------------------------------------------ resident decode (decode_resident.hip)
struct ResidentCtl {
    unsigned done;  // steps of the generation that are finished
    unsigned rest_steps, rest_members;  // steps that decode_rest_kernel has run since the handle was made, workgroups it last had
    unsigned pad[29];
    // zeroed in front of every launch
    unsigned reg[8];  // workgroups registered by XCD
    unsigned total;   // in all
    unsigned state;   // 0 open, 1 committed: all workgroups are resident, 2 withdrawn
    unsigned joined, members, arrived;  // decode_rest_kernel: workgroups that came, those that share the work, arrivals at its barriers
    unsigned pad2[19];
    unsigned passed[8][32];  // its barriers that are complete, a line for every XCD
};
struct ResidentArgs {
    // layer 0; the others lie w_stride / kv_stride bytes apart
    const void *c_attn_w, *c_proj_w, *c_fc_w, *mlp_proj_w;
    const float *ln_1_g, *c_attn_c2, *c_attn_c3, *c_proj_b, *ln_2_g, *c_fc_c2, *c_fc_c3, *mlp_proj_b;
    size_t w_stride, kv_stride;
    char *k_cache, *v_cache;  // fp32, [head][ctx][64]
    const void *wte, *wpe;
    const float *ln_f_g, *ln_f_b, *lm_c2, *lm_c3;
    int n_layer, n_heads, ctx, vocab;
    int batch;
    int n_prompt, s0, s1;  // (shortest) prompt; steps s0 .. s1 - 1 of the generation
    const int *prompt, *prompt_len;  // prompts and tokens: out_stride apart
    int out_stride;
    int *out_tokens, *cur_token;
    StepCtrl* ctrl;
    float *x, *logits, *part_val;
    int* part_idx;
    int n_part;
    unsigned long long* words;  // resident_words(n_embed, batch), zeroed once; tags tag0 .. tag0 + (s1 - s0) (n_layer + 2) - 1 are this launch's alone
    ResidentCtl* ctl;
    unsigned tag0;
    unsigned spin_limit, start_limit;
    unsigned *fault, *withdrawn;  // pinned host words
};
bool resident_shape(size_t n_embed, size_t n_heads, size_t ctx, size_t n_layer, size_t vocab);
size_t resident_words(size_t n_embed, size_t batch);
int launch_decode_resident(const ResidentArgs& a, int n_embed, int weight_type, hipStream_t s);  // one sequence: bf16 or fp32 weights; two to eight: bf16
size_t resident_batch_words(size_t n_embed);
int launch_decode_resident_batch(const ResidentArgs& a, int n_embed, hipStream_t s);
// the steps from ctl->done to s1 - 1 where launches were withdrawn (decode_rest.hip); any shape with 64 channels a head
struct RestArgs {
    ResidentArgs r;
    int n_embed;
    float *q, *z, *h;  // [batch][n_embed], [batch][n_embed], [batch][4 n_embed]
    float* best_v;     // decode_rest_floats() in all
    int* best_i;
    unsigned patience;  // polls of the first workgroup, about a microsecond each, while not all have started
};
size_t decode_rest_floats();
int launch_decode_rest(const RestArgs& a, int weight_type, hipStream_t s);

// ------------------------------------------------------------------------------------ multi-GPU (dist.hip)
int dist_broadcast(void* buf, size_t bytes, int root, hipStream_t s);  // in place, over the communicator of zg_dist_init

// ------------------------------------------------------------------------------------ decode prefetcher (prefetch.hip)
enum PfKind { PF_NONE = 0, PF_WEIGHTS = 1, PF_KV = 2 };
constexpr unsigned PF_STOP = 0xffffffffu;  // value of the progress word that ends the prefetcher
// What launch `index` of a decode step reads: weights = n_wg contiguous tiles of wg_bytes (block b reads tile b);
// KV = the rows of earlier positions of one layer's caches, laid out for the (heads, splits, batch) attention grid.
struct PfJob {
    const char* base;
    const char* base2;    // PF_KV: the V cache
    size_t total_bytes;   // PF_WEIGHTS: end of the matrix (the last tile may be short)
    unsigned wg_bytes, n_wg;
    unsigned touch_bytes;  // PF_WEIGHTS: leading part of every tile that is fetched (the whole tile unless the matrix is far larger than the L2s)
    unsigned kind;
    unsigned n_heads, ctx, batch, row_bytes;  // PF_KV
    unsigned cls;          // kernel class of the launch (1 c_attn .. 6 lm_head, as in zg_gpt_profile_step)
    unsigned pad;
    // small per-row / per-column vectors every block reads a few lines of (bias, folded-LayerNorm vectors, ln gain):
    // fetched whole into every XCD — once the weights come from the L2 these are what a block would wait for
    const char* aux[3];
    unsigned aux_bytes[3];
    unsigned pad2;
};
struct alignas(8) PfCtl {
    unsigned progress;    // (T << 8) | launches started in the step at sequence length T;  PF_STOP ends the prefetcher
    unsigned base_xcd;    // 0x100 | XCC_ID of block 0 of the step's launches (block b then runs on XCD (base + b) % 8);
                          // written with `progress` as one 64-bit store by the embed kernel
    unsigned sink_guard, sink;
    unsigned ticket[8];       // prefetcher workgroups that found themselves on XCD x
    unsigned exit_reason[8];  // 1 stop, 2 idle limit
    unsigned jobs_done[8];
    unsigned xcd_log[256];    // -DZG_STAMPS builds: 0x100 | XCC_ID of block 0 of launch i of the last step
};
struct PfArgs {
    PfCtl* ctl;
    const PfJob* jobs;  // [njobs]: index 0 = the embed kernel (nothing to fetch), then the step's launches in order
    int njobs;          // launches of a step with lm_head
    int lead;           // launches ahead of the running one
    int nsub;           // prefetcher workgroups per XCD
    int max_T;          // last sequence length of the generation (nothing is fetched for steps beyond it)
    unsigned idle_limit;
    unsigned sleep;     // s_sleep(8) repetitions between polls
    unsigned cls_mask;  // bit c set: launches of class c are fetched for
    unsigned line_shift;  // log2 of the touch stride in bytes (7 = one load per 128-byte line)
    unsigned cap_bytes;   // most bytes fetched for one launch (the head of every tile when the matrix is larger); 0 = no cap
};
int launch_prefetcher(const PfArgs& a, hipStream_t s);

// Every decode kernel counts itself in at entry (one lane of block 0; fire and forget).
__device__ __forceinline__ void pf_count(unsigned* progress) {
    if (progress != nullptr && (blockIdx.x | blockIdx.y | blockIdx.z | threadIdx.x) == 0) {
#ifdef ZG_STAMPS
        const unsigned old = __hip_atomic_fetch_add(progress, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        reinterpret_cast<PfCtl*>(progress)->xcd_log[old & 255u] = 0x100u | (__builtin_amdgcn_s_getreg((3 << 11) | 20) & 15u);
#else
        __hip_atomic_fetch_add(progress, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#endif
    }
}

}  // namespace zg
