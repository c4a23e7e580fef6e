// khq_internal.h -- kernel argument blocks and launch helpers shared by the
// kernels (khq_kernels.hip) and the C ABI layer (khq_capi.cpp).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include <atomic>

namespace khq {

// The token of a decode step, to be appended to ring slot `slot` (rows
// [h_kv][256]) by the launch that attends over it; k = NULL: none, u / ring_u
// may be NULL.
struct RingNew {
    const __half* k;
    const __half* v;
    const __half* u;
    __half* ring_k;
    __half* ring_v;
    __half* ring_u;
    int slot;
};

// Compressed-region work: token range [0, c_len) of KV head blockIdx.y cut
// into n_parts parts; the partial triple of query qid, part i lands at
// part[(qid * part_stride + part_offset + i) * 258].
struct AttnArgs {
    const __half* q;  // q_gate [H_q][512]
    const uint8_t* kpay;
    const uint8_t* vpay;
    const uint8_t* vsm;
    const uint32_t* kmask;
    const __half* knorm;
    const __half* krn;
    const __half* vnorm;
    const __half* vrn;
    const __half* cents_k;
    const __half* cents_v;
    const __half* vq;
    const __half* rotor_k;
    const __half* rotor_v;
    const __half* dk;
    const __half* dv;
    float* part;
    int c_len, h_kv, L_q, start_pos, n_parts, part_stride, part_offset;
    float sc, a_k, a_v, rope_base;
    // Optional raw ring window, computed by one extra block of the
    // wavefront-specialised kernel into partial part_offset + n_chunks
    // (win_len = 0: none).
    const __half* ring_k;
    const __half* ring_v;
    int win_start, win_len, ring_cap;
    RingNew add;     // appended by the window blocks before they read the window
    int win_blocks;  // window blocks after the chunks: 4 (one per KV head) or 1 (all heads)
    int chunk_tiles;  // batched launch: tiles per compressed chunk of this sequence
    // Bound of the key / value hand-off waits of the wavefront-specialised
    // kernel, in sleeps (set by the launchers; a test knob may lower it).
    int spin_limit;
    // Reference split partition (wavefront-specialised kernel): split_per > 0
    // cuts [0, c_len) into splits of split_per tokens, each into split_subs
    // chunks of tiles_per_chunk tiles; chunk = split * split_subs + sub.
    // split_per = 0: chunk i covers tiles [i * tiles_per_chunk, + tiles_per_chunk).
    int split_per, split_subs;
    // RoPE table of the wavefront-specialised kernel, [lane group g][3][u]:
    // freq of dim pair m = 16 (u / 4) + 4 g + u % 4, cos and sin of 16 freq
    // (filled by the launchers from rope_base).
    float rope_tab[96];
};

// fp16 ring-window work, same partial layout (query = head).
struct WinArgs {
    const __half* q;
    const __half* ring_k;
    const __half* ring_v;
    float* part;
    int win_start, win_len, ring_cap, h_kv, n_parts, part_stride, part_offset;
    float sc;
};

// Window attention + merge with compressed partials + gate (fused step tail).
// Compressed partial i of query head h at part[(h * part_stride + i) * 258].
struct FinishArgs {
    const float* part;
    int n_parts, part_stride;
    const __half* q;  // q_gate [H_q][512]
    const __half* ring_k;
    const __half* ring_v;
    int win_start, win_len, ring_cap, h_kv, n_rep;
    float sc, eps;
    __half* out;  // [H_q][256]
};
hipError_t launch_step_finish(const FinishArgs& a, int H_q, hipStream_t st);
// n_seq sequences, args a device array; the window must already be a part
// (win_len = 0 in every FinishArgs).
// Copies bytes (a multiple of 16) from pinned host memory to device memory
// with a one-block kernel on st.
hipError_t launch_meta_upload(const void* host_src, void* dst, size_t bytes, hipStream_t st);
// max_parts: the largest part count of a sequence.
hipError_t launch_step_finish_batched(const FinishArgs* args, int n_seq, int H_q, int max_parts,
                                      hipStream_t st);

// Rows of 256 halves to compress: the first n_ring from a ring buffer of
// ring_rows rows starting at row ring_row0 (wrapping), the rest from src.
struct RowSrc {
    const __half* src;
    const __half* ring;
    int n_ring, ring_row0, ring_rows;
    __device__ __forceinline__ const __half* row(int r) const {
        if (r >= n_ring) return src + (size_t)(r - n_ring) * 256;
        const int s = ring_row0 + r;
        return ring + (size_t)(s >= ring_rows ? s - ring_rows : s) * 256;
    }
};
// One compressor job.
struct CompressJob {
    RowSrc x;
    const __half* d_vec;
    const __half* rotor;
    const __half* cents;
    const __half* vq;
    uint32_t* out_mask;
    __half* out_norms;
    __half* out_rn;
    uint8_t* out_pay;
    uint8_t* out_sm;
    int n;
    float ts, alpha;
};
// The K and V jobs of one compression event in one launch.
hipError_t launch_compress_pair(const CompressJob& k, const CompressJob& v, hipStream_t st);
hipError_t launch_compress(const CompressJob& job, int is_v, hipStream_t st);
// Whether a launch over n rows uses the several-rows-a-wavefront form.
bool compress_v_many(int n);
bool compress_k_many(int n);
hipError_t launch_attn_parts(const AttnArgs& a, int n_rep, dim3 grid, hipStream_t st);
// waves: wavefronts per block, 1 or 4.
hipError_t launch_window_parts(const WinArgs& a, int n_rep, int h_kv, int waves, hipStream_t st);
hipError_t launch_lse_reduce(const float* part, float* out, int n_q, int n_parts,
                             hipStream_t st);
// subs chunk triples per split -> split triples -> their merge (splits * subs <= 256).
hipError_t launch_split_reduce(const float* part, float* out_partial, float* out, int n_q,
                               int splits, int subs, hipStream_t st);
hipError_t launch_combine_gate(const float* part, const __half* q_gate, __half* out, int H_q,
                               int n_parts, float eps, hipStream_t st);
hipError_t launch_merge_gate(const float* ac, const float* aw, const __half* qg, __half* out,
                             int H_q, int D, int has_w, hipStream_t st);
hipError_t launch_gather_q(const __half* qg, __half* qo, int H_q, int D, hipStream_t st);
hipError_t launch_ring_write(__half* rk, __half* rv, __half* ru, const __half* k,
                             const __half* v, const __half* ku, int kv, hipStream_t st);
hipError_t launch_partial_rope(__half* vec, int num_heads, int head_dim, int rotary_dim, int pos,
                               float theta, int stride, hipStream_t st);

// Compressed-region kernel for H_kv = 4, n_rep = 6, L_q = 1 (wavefront-
// specialised, 512 threads per block): one block per chunk of
// tiles_per_chunk 16-token tiles; partial index = part_offset + chunk.
int attn_ws_tiles_per_chunk(int c_len, int* n_chunks);
// Device fault word of the wavefront-specialised kernel (nonzero after a
// hand-off wait gave up), read with a synchronous copy; clear resets it.
hipError_t fault_status(int* out, int clear);
// Hand-off wait bound used by the launchers (default 2^20 sleeps).
extern std::atomic<int> g_spin_limit;
size_t attn_ws_smem_bytes();
// Whether khq_attn_step_fp16 computes this step's window inside the
// compressed-region launch (which can then append the step's token to the ring).
bool step_window_in_ws(int H_q, int H_kv, int c_len, int win_len);
// khq_attn_step_fp16 with the token of the step appended first; only where
// step_window_in_ws holds.
int attn_step_append(const AttnArgs& a, int H_q, __half* out, hipStream_t stream);
// Fills a.rope_tab from a.rope_base (host).
void fill_rope_table(AttnArgs& a);
hipError_t launch_attn_ws(const AttnArgs& a, int tiles_per_chunk, int n_chunks,
                          hipStream_t st);
// Batched: args[seq] (device) with n_parts = that sequence's chunk count and
// its window fields; map[b] = (seq, chunk) for each of n_blocks blocks (chunk
// == n_parts: the sequence's window block).
hipError_t launch_attn_ws_batched(const AttnArgs* args, const int2* map, int n_blocks,
                                  hipStream_t st);

// Head RMSNorm + unroped capture + partial RoPE + ring writes of one token
// (D = 256, rot <= 64): q_gate [H_q][512] and k [H_kv][256] in place.
struct NormRopeArgs {
    __half* q_gate;
    __half* k;
    const __half* v;
    const float* q_w;  // [256] or NULL
    const float* k_w;  // [256] or NULL
    __half* ring_k;
    __half* ring_v;
    __half* ring_u;
    int H_q, H_kv, slot, pos, rot;
    float eps, theta;
};
hipError_t launch_norm_rope(const NormRopeArgs& a, hipStream_t st);

// ---- chunked prefill (khq_prefill.hip)
// Compressed rows [tok0, tok0 + n_tok) of every KV head -> dense fp16 roped K
// rows out_k[(key0 + t) * h_kv + h][256] and V^T out_vt[h][256][ld_vt]
// columns key0 + t (ld_vt >= key0 + n_tok rounded up to 64, multiple of 8).
struct DecompArgs {
    const uint8_t* kpay;
    const uint8_t* vpay;
    const uint8_t* vsm;
    const uint32_t* kmask;
    const __half* knorm;
    const __half* krn;
    const __half* vnorm;
    const __half* vrn;
    const __half* cents_k;
    const __half* cents_v;
    const __half* vq;
    const __half* rotor_k;
    const __half* rotor_v;
    const __half* dk;
    const __half* dv;
    __half* out_k;
    __half* out_vt;
    int h_kv, tok0, n_tok, start_pos, key0, ld_vt;
    float a_k, a_v, rope_base;
    float freq[32];  // rope_base^(-2 i / 64), filled by the launchers
};
// n raw tokens (rows token * h_kv + head of k / v) -> the same key layout at
// key0 + t (key0 a multiple of 32; V^T columns up to the next multiple of 32
// are written too).
struct GatherArgs {
    RowSrc k, v;
    __half* out_k;
    __half* out_vt;
    int h_kv, n, key0, ld_vt;
};
// Division of any 32-bit n by a launch constant d: multiply and shift (Granlund
// and Montgomery, 1994).  A block's index arithmetic is on the scalar unit with
// it; the compiler's division by a variable is some 25 vector instructions.
struct FastDiv {
    uint32_t d, mul;
    int s1, s2;
    FastDiv() = default;
    explicit FastDiv(uint32_t d_) : d(d_) {
        int l = 0;
        while (l < 32 && ((uint64_t)1 << l) < d) l++;
        mul = (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << l) - d)) / d + 1);
        s1 = l < 1 ? l : 1;
        s2 = l > 1 ? l - 1 : 0;
    }
    __host__ __device__ int div(uint32_t n) const {
        const uint32_t t = (uint32_t)(((uint64_t)mul * n) >> 32);
        return (int)((t + ((n - t) >> s1)) >> s2);
    }
};
// n tokens of src_k / src_v / src_u [t][h_kv][256] -> ring slots
// (slot0 + t) % ring_cap (n <= ring_cap).
struct RingArgs {
    const __half* src_k;
    const __half* src_v;
    const __half* src_u;
    __half* ring_k;
    __half* ring_v;
    __half* ring_u;
    int h_kv, n, slot0, ring_cap;
    FastDiv by_token;  // 8-byte pieces per token, filled by the launcher
};
// n_q queries (q_gate rows [n_q][H_q][512]) over two runs of dense keys:
// decoded tokens at key indices [0, ..) and raw tokens at raw0 + r, r < n_raw
// (raw0 a multiple of 32).  Query j has seen vis = min(n_raw, vis0 + j) raw
// tokens; of these the first bound(vis), a multiple of 128, have been
// compressed by then, so it attends to decoded keys [0, dec0 + bound(vis)) and
// raw keys [bound(vis), vis).  bound follows the ring: none below 256, then
// 128 more every 128 tokens, at most ev_cap (dec0 and ev_cap multiples of
// 128; ev_cap = 0: every key is raw).
// Rows of one KV head (query j, head r % n_rep) are cut into blocks, a block's
// 32-key tiles into ceil(tiles / unit) splits (at most n_split; with uniform, into
// n_split).  Blocks of one split write out directly unless apart; split s of the
// others leaves the triple of (query j, head hq) at
// part[((j * H_q + hq) * n_split + s) * 258].
struct PrefillArgs {
    const __half* q;
    const __half* k;
    const __half* vt;
    float* part;
    __half* out;  // NULL: triples only (apart)
    int ld_vt, n_q, h_kv, n_rep, n_split;
    int round_up;  // unit - 1, or with uniform what makes by_unit's quotient n_split
    bool apart;    // every block leaves triples
    bool uniform;  // every block has n_split splits
    int vis0, n_raw, raw0, dec0, ev_cap;
    float sc, eps;
    FastDiv by_rep, by_hq, by_kv, by_split, by_unit;  // n_rep, H_q, h_kv, n_split, unit
    int unit;  // tiles of a split
    __host__ __device__ int bound(int vis) const {
        if (ev_cap <= 0 || vis < 256) return 0;
        const int b = (((vis - 256) >> 7) + 1) << 7;
        return b < ev_cap ? b : ev_cap;
    }
    __host__ __device__ int vis_of(int j) const { return vis0 + j < n_raw ? vis0 + j : n_raw; }
    // Tiles of a block of rows [row_first, row_last]: tile i is decoded tile i
    // for i < nd, then raw tile u0 + i - nd.
    __host__ __device__ int block_tiles(int row_first, int row_last, int* nd, int* u0) const {
        const int vf = vis_of(by_rep.div(row_first)), vl = vis_of(by_rep.div(row_last));
        *nd = (dec0 + bound(vl)) >> 5;
        *u0 = bound(vf) >> 5;
        return *nd + ((vl + 31) >> 5) - *u0;
    }
    __host__ __device__ int block_splits(int tiles) const { return by_unit.div(tiles + round_up); }
    size_t triple_bytes(int splits) const {
        return (size_t)n_q * h_kv * n_rep * splits * 258 * sizeof(float);
    }
};
hipError_t launch_decompress(const DecompArgs& a, hipStream_t st);
hipError_t launch_ring_gather(const GatherArgs& a, hipStream_t st);
// A decode and a gather whose outputs are disjoint, in one launch.
hipError_t launch_decompress_gather(const DecompArgs& d, const GatherArgs& g, hipStream_t st);
// A compression event (k, v: rows (token, KV head) of the chunk), the decode
// of those rows (d: tok0 = key0, n_tok tokens, start_pos 0) and a gather
// (disjoint from the decoded rows) in one launch.
hipError_t launch_compress_decode(const CompressJob& k, const CompressJob& v, const DecompArgs& d,
                                  const GatherArgs& g, hipStream_t st);
// Several events' rows and a gather in one launch (no decode).
hipError_t launch_compress_gather(const CompressJob& k, const CompressJob& v, const GatherArgs& g,
                                  hipStream_t st);
// Rows of one KV head a block of the prefill attention takes.
int prefill_block_rows(int n_rows);
// Fills a.n_split, a.unit, a.apart and a.uniform for the current device, the
// triples in at most max_bytes where that is possible.
void prefill_plan(PrefillArgs& a, size_t max_bytes);
hipError_t launch_prefill_attn(const PrefillArgs& a, hipStream_t st);
// Prefill attention plus merge and gate through the shared workspace: q, k, vt,
// the shapes, the key runs and out set in a; with ring, its copy runs behind
// the attention.  merge = false: the attention launch alone, every block's
// triples left in the workspace.
int prefill_attn_run(PrefillArgs a, const RingArgs* ring, hipStream_t stream, bool merge = true);
// Merge of the split blocks' triples, / (den + eps), sigmoid gate from q_gate
// row r (gate at 256..511), and the ring copy (ring may be NULL), in one launch.
hipError_t launch_prefill_finish(const PrefillArgs& a, const RingArgs* ring, hipStream_t st);

// Per-device launch set-up, cached per device index under a lock (a process
// may drive several GPUs from several threads): the CU count of the current
// device, and the dynamic-LDS limit of a kernel raised to `bytes` on the
// current device (once per (kernel, device)).
int device_cu_count();
hipError_t ensure_dynamic_lds(const void* kernel, int bytes);

}  // namespace khq
