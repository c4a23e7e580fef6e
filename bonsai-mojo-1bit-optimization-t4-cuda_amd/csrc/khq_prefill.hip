// khq_prefill.hip -- chunked prefill on matrix cores: many query tokens of one
// layer attend to the compressed prefix and the raw ring window at once.
//
// Kernels that build one dense fp16 key space (key index = token position)
// and attend over it causally:
//   decompress_kernel   compressed rows -> roped K rows [key][H_kv][256] and
//                       V^T [H_kv][256][ld] (the decode of the compressed-
//                       region attention kernel, ref:src/csrc/
//                       qmv_sm75_kernel.cu:1608-1699 for K and :1739-1762,
//                       1776-1826 for V, applied per token instead of being
//                       folded into the running sums);
//   ring_gather_kernel  raw tokens (ring slots, then the caller's) -> K rows
//                       and V^T columns of the raw run;
//   compress_decode_kernel  a compression event that decodes the rows it
//                       packs into the key space (and gathers raw tokens);
//   compress_gather_kernel  many events' rows (and the gather);
//   prefill_attn_kernel, prefill_attn_rs_kernel  S^T = K Q^T and
//                       O^T = V^T P^T on MFMA (fp16 in, fp32 accumulate),
//                       online softmax, one split of a block's keys per block;
//   prefill_finish_kernel  the splits' partial triples merged and gated, the
//                       new tokens copied to their ring slots.
// One launch serves queries on both sides of any number of compression events:
// a block walks the decoded tiles its last query sees, then the raw tiles from
// its first query's compressed bound on, and each row masks what it does not
// see (PrefillArgs).
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <cmath>

#include "khq_internal.h"
#include "khq_mfma_util.h"
#include "khq_decode_row.h"
#include "khq_compress_row.h"

namespace khq {
namespace pf {

using namespace mu;

constexpr int BLK_THR = 256;  // decompress / gather blocks: 4 wavefronts of TB / 4 tokens
constexpr int VT_PAD = 8;     // halves of padding per LDS V^T row
// Tokens per block TB: 4 spread a chunk over many CUs; 16 write V^T in 32-byte
// runs and set a lane's constants up once for four tokens, but take 12 us
// however few there are.
constexpr int TB_LONG = 16;

// Writes columns [0, nc) of the block's LDS V^T tile (nc <= TB a multiple of 4)
// to vt columns key0 .. of KV head h, in pieces of 8 bytes (TB 4) or 16.
template <int TB>
__device__ __forceinline__ void store_vt(const _Float16 (*sv)[TB + VT_PAD], __half* vt, int ld,
                                         int h, int key0, int nc) {
    constexpr int W = TB < 8 ? 4 : 8;  // columns per piece
    for (int i = threadIdx.x; i < 256 * (TB / W); i += BLK_THR) {
        const int d = i / (TB / W), c = i % (TB / W) * W;
        __half* dst = vt + ((size_t)h * 256 + d) * ld + key0 + c;
        if (W == 8 && c + 8 <= nc)
            *reinterpret_cast<u4q*>(dst) = *reinterpret_cast<const u4q*>(&sv[d][c]);
        else if (c < nc)
            *reinterpret_cast<uint2*>(dst) = *reinterpret_cast<const uint2*>(&sv[d][c]);
    }
}

// ------------------------------------------------------------- decompress
// Block (TB tokens, KV head h), a wavefront per TB / 4 tokens; lane p owns
// patch p = dims 4 p .. 4 p + 3.  Latency-bound: the decode of a row is a chain
// of dependent reads (mask -> ordinals -> payload bytes, fields -> codebook), so
// the block's packed rows come to LDS in one round trip first, and every
// token's codebook entry is requested before the first row is decoded.
// 8,000 rows 21.9 -> 15.8 us, 512 rows 7.1 -> 5.9 us, 130,560 rows 227 -> 121 us.
template <int TB>
using VtTile = _Float16[256][TB + VT_PAD];
template <int TB>
struct __align__(16) DecompLds {
    VtTile<TB> sv;
    uint32_t pay[TB][53];  // mask 16 words, K payload 10, V payload 26
    float nrm[TB][5];      // K norm, residual scale; V norm, energy, shared meta
};
template <int TB>
__device__ __forceinline__ void decompress_block(const DecompArgs& a, int bx, int h, void* lds) {
    DecompLds<TB>& L = *static_cast<DecompLds<TB>*>(lds);
    auto& sv = L.sv;
    const int wv = threadIdx.x >> 6, p = threadIdx.x & 63;
    const int t_blk = bx * TB;
    auto row_of = [&](int tl) { return (size_t)(a.tok0 + min(t_blk + tl, a.n_tok - 1)) * a.h_kv + h; };
#pragma unroll
    for (int i0 = 0; i0 < TB * 52; i0 += BLK_THR) {
        const int i = i0 + threadIdx.x, tl = i / 52, w = i % 52;
        if (i < TB * 52) {
            const size_t g = row_of(tl);
            const u1b* src = w < 16   ? reinterpret_cast<const u1b*>(a.kmask + g * 16) + w
                             : w < 26 ? reinterpret_cast<const u1b*>(a.kpay + g * 40) + w - 16
                                      : reinterpret_cast<const u1b*>(a.vpay + g * 104) + w - 26;
            L.pay[tl][w] = *src;
        }
    }
    if (threadIdx.x < TB * 5) {
        const int tl = threadIdx.x / 5, f = threadIdx.x % 5;
        const size_t g = row_of(tl);
        const __half* n = f == 0 ? a.knorm : f == 1 ? a.krn : f == 2 ? a.vnorm : a.vrn;
        L.nrm[tl][f] = f == 4 ? __uint_as_float(*reinterpret_cast<const u1b*>(a.vsm + g * 4))
                              : __half2float(n[g]);
    }
    dec::Consts cs;
    dec::load_consts(a, p, cs);
    __syncthreads();
    constexpr int TW = TB / 4;  // tokens per wavefront: wv, wv + 4, ...
    uint32_t fld[TW];
    float cbv[TW][3];
    const uint32_t grp = (uint32_t)p / 8, bit = 12 * ((uint32_t)p % 8);
#pragma unroll
    for (int i = 0; i < TW; i++) {
        const uint32_t* vw = &L.pay[wv + 4 * i][26];
        const uint32_t w = grp * 3 + (bit >> 5);  // (the words after the fields are there)
        fld[i] = __builtin_amdgcn_alignbit(vw[w + 1], vw[w], bit & 31) & 0xFFFu;
        const uint32_t code = (fld[i] & 0x7Fu) | (((vw[24 + (p >> 5)] >> (p & 31)) & 1u) << 7);
#pragma unroll
        for (int k = 0; k < 3; k++) cbv[i][k] = __half2float(a.vq[(size_t)p * 768 + code * 3 + k]);
    }
#pragma unroll
    for (int i = 0; i < TW; i++) {
        const int tl = wv + 4 * i, tok = t_blk + tl;
        const bool ok = tok < a.n_tok;  // uniform per wavefront
        const float* nr = L.nrm[tl];
        float y[4];
        // ---- K: codes, outlier ordinals (ballot prefix), values, RoPE
        dec::decode_k(a, cs, L.pay[tl][p >> 2], reinterpret_cast<const uint8_t*>(&L.pay[tl][16]), nr[0],
                      nr[1], (float)(a.start_pos + a.tok0 + tok), p, y);
        if (ok)
            *reinterpret_cast<uint2*>(a.out_k + ((size_t)(a.key0 + tok) * a.h_kv + h) * 256 + 4 * p) =
                uint2{pk_rne(y[0], y[1]), pk_rne(y[2], y[3])};
        // ---- V: codebook, dim 3, inverse rotor, FWHT
        dec::decode_v_cb(a, cs, cbv[i], fld[i], nr[2], nr[3], nr[4], p, y);
#pragma unroll
        for (int c = 0; c < 4; c++) sv[4 * p + c][tl] = ok ? (_Float16)y[c] : (_Float16)0.0f;
    }
    __syncthreads();
    store_vt<TB>(sv, a.out_vt, a.ld_vt, h, a.key0 + t_blk, min(TB, (a.n_tok - t_blk + 3) & ~3));
}

// ------------------------------------------------------------- raw gather
// Block (32 raw tokens, KV head h), eight a wavefront: K rows copied, V rows
// transposed through LDS, every row of the block in flight at once.  Tokens past
// the last give zero V^T columns.  A lane's eight tokens go to LDS as one 16-byte
// piece a dim: as single halves (32 stores a lane, 32 lanes to a bank) they took
// 1.7 us of a short prompt.
__device__ __forceinline__ void gather_block(const GatherArgs& a, int bx, int h, void* lds) {
    VtTile<32>& sv = *static_cast<VtTile<32>*>(lds);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int t0 = bx * 32 + wv * 8;
    uint2 kw[8], vw[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int r = min(t0 + i, a.n - 1) * a.h_kv + h;
        kw[i] = *reinterpret_cast<const uint2*>(a.k.row(r) + 4 * lane);
        vw[i] = *reinterpret_cast<const uint2*>(a.v.row(r) + 4 * lane);
    }
    h8 col[4];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int t = t0 + i;
        if (t < a.n)
            *reinterpret_cast<uint2*>(a.out_k + ((size_t)(a.key0 + t) * a.h_kv + h) * 256 + 4 * lane) =
                kw[i];
        const h4 v = __builtin_bit_cast(h4, t < a.n ? vw[i] : uint2{0u, 0u});
#pragma unroll
        for (int c = 0; c < 4; c++) col[c][i] = v[c];
    }
#pragma unroll
    for (int c = 0; c < 4; c++) *reinterpret_cast<h8*>(&sv[4 * lane + c][8 * wv]) = col[c];
    __syncthreads();
    store_vt<32>(sv, a.out_vt, a.ld_vt, h, a.key0 + bx * 32, 32);
}
// Flat block index of a gather: token block fastest, then the KV head.
__device__ __forceinline__ void gather_flat(const GatherArgs& a, int b, void* lds) {
    const int nx = (a.n + 31) / 32;
    gather_block(a, b % nx, b / nx, lds);
}
// LDS of a launch whose blocks do one of several jobs: the largest job's.
template <size_t... N>
struct __align__(16) SharedLds {
    static constexpr size_t bytes = std::max({N...});
    unsigned char b[bytes];
};

template <int TB>
__global__ __launch_bounds__(BLK_THR) void decompress_kernel(DecompArgs a) {
    __shared__ SharedLds<sizeof(DecompLds<TB>)> lds;
    decompress_block<TB>(a, blockIdx.x, blockIdx.y, &lds);
}

__global__ __launch_bounds__(BLK_THR) void ring_gather_kernel(GatherArgs a) {
    __shared__ SharedLds<sizeof(VtTile<32>)> lds;
    gather_flat(a, blockIdx.x, &lds);
}

// A decode and an independent gather (disjoint outputs, no data passed
// between them) in one launch: blocks [0, nx_d h_kv) decode (x fastest, then
// the KV head), the rest gather.
template <int TB>
__global__ __launch_bounds__(BLK_THR) void decompress_gather_kernel(DecompArgs d, GatherArgs g,
                                                                    int nx_d) {
    __shared__ SharedLds<sizeof(DecompLds<TB>), sizeof(VtTile<32>)> lds;
    const int nb_d = nx_d * d.h_kv, b = blockIdx.x;
    if (b < nb_d)
        decompress_block<TB>(d, b % nx_d, b / nx_d, &lds);
    else
        gather_flat(g, b - nb_d, &lds);
}

// A compression event, the decode of its rows into the dense key space and
// the raw gather in one launch: blocks [0, nb_k) compress and decode K rows
// (four per block, the longest blocks, first), [nb_k, nb_k + n_v) V rows (one
// per block), the rest gather.
__global__ __launch_bounds__(BLK_THR) void compress_decode_kernel(CompressJob k, CompressJob v,
                                                                  DecompArgs d, GatherArgs g,
                                                                  int nb_k) {
    __shared__ SharedLds<sizeof(CompressLds), sizeof(VtTile<32>)> lds;
    int b = blockIdx.x;
    if (b < nb_k) {
        compress_block<true>(k.x, k.d_vec, k.rotor, k.cents, k.vq, k.out_mask, k.out_norms,
                             k.out_rn, k.out_pay, nullptr, k.n, k.ts, k.alpha, 0, b, &lds, &d);
        return;
    }
    b -= nb_k;
    if (b < v.n) {
        compress_block<true>(v.x, v.d_vec, v.rotor, v.cents, v.vq, v.out_mask, v.out_norms,
                             v.out_rn, v.out_pay, v.out_sm, v.n, v.ts, v.alpha, 1, b, &lds, &d);
        return;
    }
    gather_flat(g, b - v.n, &lds);
}

// The rows of several compression events and the raw gather in one launch:
// K blocks (four rows each, or 4 KR with k_many), V blocks (VR rows), gather.
__global__ __launch_bounds__(BLK_THR) void compress_gather_kernel(CompressJob k, CompressJob v,
                                                                  GatherArgs g, int nb_k, int nb_v,
                                                                  int k_many) {
    __shared__ SharedLds<sizeof(CompressLds), sizeof(VRowsLds), sizeof(KRowsLds), sizeof(VtTile<32>)> lds;
    int b = blockIdx.x;
    if (b < nb_k) {
        if (k_many)
            compress_k_rows(k, b, &lds);
        else
            compress_block(k.x, k.d_vec, k.rotor, k.cents, k.vq, k.out_mask, k.out_norms, k.out_rn,
                           k.out_pay, nullptr, k.n, k.ts, k.alpha, 0, b, &lds);
        return;
    }
    b -= nb_k;
    if (b < nb_v)
        compress_v_rows(v, b, &lds);
    else
        gather_flat(g, b - nb_v, &lds);
}

// Visibility of the keys of one 32-key tile to one query row, as a bit mask
// (bit i: key i of the tile): a decoded tile lies wholly below or wholly at or
// past the row's compressed bound (both are multiples of 32), a raw tile wholly
// before it or up to the row's causal end.  Only vis and the bound stay live.
__device__ __forceinline__ uint32_t bits_below(int n) {  // bits [0, n) of 32
    return n >= 32 ? ~0u : (n <= 0 ? 0u : (1u << n) - 1u);
}
struct RowKeys {
    int vis, bnd, dec_end;
    __device__ __forceinline__ RowKeys(const PrefillArgs& a, int jq)
        : vis(a.vis_of(jq)), bnd(a.bound(a.vis_of(jq))), dec_end(0) {
        dec_end = a.dec0 + bnd;
    }
    // dec: decoded tile; base: its first token (decoded) or raw index
    __device__ __forceinline__ uint32_t tile(bool dec, int base) const {
        // selects, no branch: a divergent branch here costs the 32-row
        // kernel about 45 registers (spilled to AGPRs)
        const int end = dec ? dec_end : vis, lo = dec ? 0 : bnd;
        const uint32_t m = bits_below(end - base);
        return base >= lo ? m : 0u;
    }
};
// The block's tile list (PrefillArgs) and this split's part of it, `per` tiles.
struct BlockKeys {
    int nd, u0, t_lo, t_hi;
    __device__ __forceinline__ BlockKeys(int nd_, int u0_, int n, int split, int per)
        : nd(nd_), u0(u0_), t_lo(min(n, split * per)), t_hi(min(n, t_lo + per)) {}
    __device__ __forceinline__ bool dec(int t) const { return t < nd; }
    __device__ __forceinline__ int base(int t) const { return 32 * (t < nd ? t : u0 + t - nd); }
};
// Longest blocks first: the last query blocks see the most keys.  Block index =
// ((reversed row block) * h_kv + head) * n_split + split.
struct BlockPos {
    int bx, h, split;
    __device__ __forceinline__ BlockPos(const PrefillArgs& a, int n_blk) {
        const int b = blockIdx.x, rest = a.by_split.div(b), rev = a.by_kv.div(rest);
        split = b - rest * a.n_split;
        h = rest - rev * a.h_kv;
        bx = n_blk - 1 - rev;
    }
};
// Row r of a KV head: its query and its head of the group.
struct RowPos {
    int j, g;
    __device__ __forceinline__ RowPos(const PrefillArgs& a, int r) : j(a.by_rep.div(r)), g(r - j * a.n_rep) {}
};

// ----------------------------------------------------------- attention
// Block = 4 wavefronts = 4 tiles of 16 query rows of one KV head, one key
// split.  Row r of KV head h is (query j = r / n_rep, head h n_rep + r % n_rep).
// Per 32-key tile the block stages K (32 x 256) and V^T (256 x 32) in LDS
// (double-buffered, one barrier per tile; the next tile's global loads are in
// flight while this one is computed), then each wavefront computes
//   S^T (two 16-key halves x 16 rows) = 16 MFMA 16x16x32, A = K rows, B = Q^T
//   (registers); lane (row li, lg) gets keys 4 lg .. 4 lg + 3 of each half;
//   O^T (256 dims x 16 rows) += 16 MFMA 16x16x32 with K = the tile's 32 keys
//   in the order (4 lg .. 4 lg + 3, 16 + 4 lg .. 16 + 4 lg + 3) per lane
//   group, so P^T is the S^T C layout as is and A = V^T read in that order.
// Softmax: a per-row reference maximum shared by the row's 4 lanes, raised
// (with a cross-lane reduction and a rescale) only when a score exceeds it by
// more than 8, so weights stay <= e^8; row sums are per lane until the end.
constexpr int KT = 32;            // keys per tile
constexpr int KS_LD = 256 + 16;   // halves per LDS K row (bank spread measured with
                                  // SQ_LDS_BANK_CONFLICT)
constexpr int VS_LD = KT + 4;     // halves per LDS V^T row (rows 8-byte aligned:
                                  // stored and read in 8-byte pieces)
constexpr float GAP = 8.0f;

// l plus both halves of a packed weight pair (fp32 sum): row sums are taken over
// the weights as the MFMAs use them, rounded to fp16, so a row's weights sum to
// one exactly as applied and one rounding error does not become two.  Rows of
// few keys gain the most; it is also half the adds.
__device__ __forceinline__ float add_pair(uint32_t pw, float l) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, pw), h2{(_Float16)1.0f, (_Float16)1.0f}, l, false);
}

// A wavefront's R rows (row0 on, of KV head h), left in LDS as floats (OUT_LD a
// row), stored a row at a time: direct rows, already divided by their sums,
// gated and rounded to the output; the others as the split's triples, with
// m / l the row's maximum and sum in lane i (< R).  Each instruction writes a
// whole row, 1 KB: the accumulators' own layout covers a 128-byte line in four
// stores of 32 bytes, and with other lines' stores between those the 32 MB of
// triples of a 128-query launch cost it 9 us more.
constexpr int OUT_LD = 260;
template <int R>
__device__ __forceinline__ void store_rows(const PrefillArgs& a, const float* so, int row0, int h, int split,
                                           bool direct, float m, float l, int lane) {
    const int n = min(R, a.n_q * a.n_rep - row0), H_q = a.h_kv * a.n_rep;
    if (n <= 0) return;  // uniform per wavefront
    const RowPos first(a, row0);
    // output row of row0 + i, stepped: within the group, then to the next query
    struct Step {
        size_t row;
        int g;
    };
    auto next = [&](Step& p) {
        const bool wrap = ++p.g == a.n_rep;
        p.row += wrap ? H_q - a.n_rep + 1 : 1;
        p.g = wrap ? 0 : p.g;
    };
    Step p{(size_t)first.j * H_q + h * a.n_rep + first.g, first.g};
    if (direct) {
        constexpr int G = 16;  // rows whose gates are in flight together
#pragma unroll 1
        for (int i0 = 0; i0 < n; i0 += G) {
            uint2 g[G];
            Step q = p;
#pragma unroll
            for (int i = 0; i < G; i++) {
                g[i] = *reinterpret_cast<const uint2*>(a.q + q.row * 512 + 256 + 4 * lane);
                if (i0 + i + 1 < n) next(q);
            }
#pragma unroll
            for (int i = 0; i < G; i++) {
                if (i0 + i >= n) break;  // uniform per wavefront
                const h4 gh = __builtin_bit_cast(h4, g[i]);
                const f4 v = *reinterpret_cast<const f4*>(&so[(i0 + i) * OUT_LD + 4 * lane]);
                float o[4];
#pragma unroll
                for (int c = 0; c < 4; c++) o[c] = v[c] * (1.0f / (1.0f + expf(-(float)gh[c])));
                *reinterpret_cast<uint2*>(a.out + p.row * 256 + 4 * lane) =
                    uint2{pk_rne(o[0], o[1]), pk_rne(o[2], o[3])};
                next(p);
            }
        }
        return;
    }
    float* part = a.part + (size_t)split * 258;
    const size_t ld = (size_t)a.n_split * 258;
    if (lane < n) {
        const RowPos r(a, row0 + lane);
        float* ml = part + ((size_t)r.j * H_q + h * a.n_rep + r.g) * ld + 256;
        ml[0] = m;
        ml[1] = l;
    }
#pragma unroll 8
    for (int i = 0; i < n; i++) {
        *reinterpret_cast<f4s*>(part + p.row * ld + 4 * lane) =
            *reinterpret_cast<const f4*>(&so[i * OUT_LD + 4 * lane]);
        next(p);
    }
}

// Grid (row block, KV head, split), the tile lists of the at most two row blocks
// worked out by the host: nothing but the arguments stands before the first
// load.  A split past its block's tiles leaves an empty triple, so every row has
// n_split of them.
struct FewBlocks {
    int nd[2], u0[2], n[2];
};
__global__ __launch_bounds__(256) void prefill_attn_kernel(PrefillArgs a, FewBlocks f) {
    __shared__ __align__(16) _Float16 ks[2][KT][KS_LD];
    __shared__ __align__(16) _Float16 vs[2][256][VS_LD];
    const int tid = threadIdx.x;
    const int wv = tid >> 6, lane = tid & 63;
    const int li = lane & 15, lg = lane >> 4;
    const int n_rows = a.n_q * a.n_rep;
    const int bx = blockIdx.x, h = blockIdx.y, split = blockIdx.z;
    const int row0 = (bx * 4 + wv) * 16;
    const int H_q = a.h_kv * a.n_rep;
    const int r = row0 + li;
    const bool r_ok = r < n_rows;
    const RowPos rp(a, r_ok ? r : 0);
    const int jq = rp.j, hq = h * a.n_rep + rp.g;
    const RowKeys vis(a, jq);
    const BlockKeys bk(f.nd[bx], f.u0[bx], f.n[bx], split, a.unit);

    h8 qb[8];
    {
        const __half* qrow = a.q + ((size_t)jq * H_q + hq) * 512;
#pragma unroll
        for (int st = 0; st < 8; st++) {
            const uint4 v = *reinterpret_cast<const uint4*>(qrow + 32 * st + 8 * lg);
            qb[st] = __builtin_bit_cast(h8, r_ok ? v : uint4{0u, 0u, 0u, 0u});
        }
    }
    f4 acc[16];
#pragma unroll
    for (int m = 0; m < 16; m++) acc[m] = f4{0.f, 0.f, 0.f, 0.f};
    float m_ref = -INFINITY, l_part = 0.0f;

    // cooperative tile loads: thread t -> K key t / 8, 64 B at (t % 8) * 32
    // halves; V^T dim t, the tile's 32 keys (64 B)
    const int ld_key = tid >> 3, ld_off = (tid & 7) * 32;
    const __half* kg = a.k + (size_t)h * 256 + ld_off;
    const __half* vg = a.vt + ((size_t)h * 256 + tid) * a.ld_vt;
    uint4 pk[4], pv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) pk[i] = pv[i] = uint4{0u, 0u, 0u, 0u};
    const int raw_end = a.raw0 + a.n_raw;
    auto key_of = [&](int t) { return (bk.dec(t) ? 0 : a.raw0) + bk.base(t); };
    auto gload = [&](int t) {
        const int k0 = key_of(t);
        const int key = bk.dec(t) ? k0 + ld_key : min(k0 + ld_key, raw_end - 1);
        const uint4* ksrc = reinterpret_cast<const uint4*>(kg + (size_t)key * a.h_kv * 256);
        const uint4* vsrc = reinterpret_cast<const uint4*>(vg + k0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            pk[i] = ksrc[i];
            pv[i] = vsrc[i];
        }
    };
    // V^T word w of a tile row holds keys 2 w, 2 w + 1; columns past the last
    // raw key are padding and become zero
    auto vmask = [](uint32_t w, int i, int nv) {
        return 2 * i + 1 < nv ? w : (2 * i < nv ? (w & 0xFFFFu) : 0u);
    };
    auto lstore = [&](int buf, int t) {
        const int nv = bk.dec(t) ? KT : a.n_raw - bk.base(t);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            *reinterpret_cast<uint4*>(&ks[buf][ld_key][ld_off + 8 * i]) = pk[i];
            uint4 v = pv[i];
            if (nv < KT)
                v = uint4{vmask(v.x, 4 * i, nv), vmask(v.y, 4 * i + 1, nv), vmask(v.z, 4 * i + 2, nv),
                          vmask(v.w, 4 * i + 3, nv)};
            *reinterpret_cast<uint2*>(&vs[buf][tid][8 * i]) = uint2{v.x, v.y};
            *reinterpret_cast<uint2*>(&vs[buf][tid][8 * i + 4]) = uint2{v.z, v.w};
        }
    };

    if (bk.t_lo < bk.t_hi) {
        gload(bk.t_lo);
        lstore(0, bk.t_lo);
        if (bk.t_lo + 1 < bk.t_hi) gload(bk.t_lo + 1);
    }
    __syncthreads();
    for (int t = bk.t_lo; t < bk.t_hi; t++) {
        const int buf = (t - bk.t_lo) & 1;
        // ---- S^T of both 16-key halves from LDS
        f4 s0 = f4{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int st = 0; st < 8; st++) {
            const h8 ka = *reinterpret_cast<const h8*>(&ks[buf][li][32 * st + 8 * lg]);
            const h8 kb = *reinterpret_cast<const h8*>(&ks[buf][16 + li][32 * st + 8 * lg]);
            s0 = mfma32(ka, qb[st], s0);
            s1 = mfma32(kb, qb[st], s1);
        }
        float sc[8], lmax = -INFINITY;
        {
            const uint32_t mb = vis.tile(bk.dec(t), bk.base(t)) >> (4 * lg);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                sc[c] = (mb >> c) & 1u ? s0[c] * a.sc : -INFINITY;
                sc[4 + c] = (mb >> (16 + c)) & 1u ? s1[c] * a.sc : -INFINITY;
            }
        }
#pragma unroll
        for (int e = 0; e < 8; e++) lmax = fmaxf(lmax, sc[e]);
        // ---- raise the row's reference maximum only when needed
        if (__ballot(lmax > m_ref + GAP) != 0ull) {
            float rmax = fmaxf(lmax, __shfl_xor(lmax, 16, 64));
            rmax = fmaxf(rmax, __shfl_xor(rmax, 32, 64));
            const float m_new = fmaxf(m_ref, rmax);
            if (m_new > m_ref) {
                const float fac = __expf(m_ref - m_new);  // 0 when m_ref = -inf
#pragma unroll
                for (int m = 0; m < 16; m++) acc[m] *= fac;
                l_part *= fac;
                m_ref = m_new;
            }
        }
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; e++) p[e] = sc[e] == -INFINITY ? 0.0f : __expf(sc[e] - m_ref);
        uint32_t pw[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            pw[e] = pk_rne(p[2 * e], p[2 * e + 1]);
            l_part = add_pair(pw[e], l_part);
        }
        const h8 pb = __builtin_bit_cast(h8, uint4{pw[0], pw[1], pw[2], pw[3]});
        // ---- O^T += V^T P^T (K = the 32 keys in the lane order above)
#pragma unroll
        for (int m4 = 0; m4 < 16; m4 += 4) {  // 4 operand reads in flight, then 4 MFMAs
            h8 vop[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint2 va = *reinterpret_cast<const uint2*>(&vs[buf][16 * (m4 + i) + li][4 * lg]);
                const uint2 vb = *reinterpret_cast<const uint2*>(&vs[buf][16 * (m4 + i) + li][16 + 4 * lg]);
                vop[i] = __builtin_bit_cast(h8, uint4{va.x, va.y, vb.x, vb.y});
            }
            __builtin_amdgcn_sched_barrier(0);  // keep the 4 reads ahead of their MFMAs
#pragma unroll
            for (int i = 0; i < 4; i++) acc[m4 + i] = mfma32(vop[i], pb, acc[m4 + i]);
        }
        // ---- stage the next tile, load the one after
        if (t + 1 < bk.t_hi) {
            lstore(buf ^ 1, t + 1);
            if (t + 2 < bk.t_hi) gload(t + 2);
        }
        __syncthreads();
    }
    // ---- row li (dims 16 mt + 4 lg + c): its triple, in the accumulators' layout
    // (a few rows: through LDS a whole row at a time takes 1 us more)
    float l_row = l_part + __shfl_xor(l_part, 16, 64);
    l_row += __shfl_xor(l_row, 32, 64);
    if (!r_ok) return;
    const bool empty = m_ref == -INFINITY;
    float* out = a.part + ((size_t)(jq * H_q + hq) * a.n_split + split) * 258;
#pragma unroll
    for (int mt = 0; mt < 16; mt++)
        *reinterpret_cast<f4s*>(out + 16 * mt + 4 * lg) = empty ? f4{0.f, 0.f, 0.f, 0.f} : acc[mt];
    if (lg == 0) {
        out[256] = empty ? -1e20f : m_ref;
        out[257] = empty ? 0.0f : l_row;
    }
}

// 32-row form: 32 query rows per wavefront pair on 32x32x16 MFMAs, so every
// K / V^T operand read from LDS feeds twice the arithmetic of the 16-row
// form; the O^T accumulators (32 rows x 256 dims) and Q^T (32 x 256 fp16)
// stay in registers, split between the pair.  32x32 layouts (lane l,
// n = l % 32, hh = l / 32):
//   A[m][k]: lane m + 32 (k / 8) holds element k % 8;  B[k][n] likewise;
//   C[m][n]: lane n + 32 hh, register r <-> m = 8 (r / 4) + 4 hh + r % 4.
// S^T = K Q^T (keys x rows); its C registers 8 s' .. 8 s' + 7 are the B
// operand of K-step s' of O^T += V^T P^T when that step's K order is
// key 8 (2 s' + i / 4) + 4 hh + i % 4 for element i, which is how V^T is read.
typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f32x16 mfma3232(h8 a, h8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
constexpr int KS2_LD = 256 + 8;   // halves per LDS K row
constexpr int VS2_LD = KT + 4;    // halves per LDS V^T row

constexpr int NKB = 3;            // LDS tile slots
// Reference of a row that has seen no key: finite, so that a masked score less
// it is -inf and its weight 0 without a test.
constexpr float M_NONE = -1e30f;
constexpr float LOG2E = 1.44269504f, LN2 = 0.693147181f;
// Lazy-rescale gap of the 32-row form, in its log2 units: weights stay <= e^10
// (< fp16 max).
constexpr float GAP32 = 10.0f * LOG2E;

// Role-specialised 32-row attention: per SIMD a score wavefront and an
// output wavefront (8 wavefronts per block, 128 rows of one KV head).  The
// score wavefront of row group g computes S^T = K Q^T (tile t + 1 on the
// matrix cores while tile t is masked, scaled and its row maximum taken),
// decides whether the row's reference maximum rises (rescale factor fac) and
// leaves tile t's masked scores with (max, fac) in LDS; the output wavefront
// of g, one tile behind, rescales its accumulators and row sums by fac,
// forms P = exp(s - max) as fp16 (the C layout of S^T is the B operand layout
// of O^T += V^T P^T) and applies the tile with 16 MFMAs.  Each role needs
// about half the registers of one wavefront doing both, so the two share a
// SIMD and one's vector work runs under the other's matrix work.  The score
// side stages the K tiles and the output side the V^T tiles in the
// three-slot ring; one block barrier per tile orders all of it (every
// wavefront passes the same barriers).
__global__ __launch_bounds__(512, 1) __attribute__((amdgpu_waves_per_eu(2, 2)))
void prefill_attn_rs_kernel(PrefillArgs a) {
    __shared__ union __align__(16) {
        struct {
            _Float16 ks[NKB][KT][KS2_LD], vs[NKB][256][VS2_LD];
            f4 pss[2][4][4][64];   // masked scaled scores (slot, row group, quad, lane)
            float2 pmf[2][4][64];  // (reference max, rescale factor) per slot
        } t;
        float out[4][32][OUT_LD];
    } lds;
    auto& ks = lds.t.ks;
    auto& vs = lds.t.vs;
    auto& pss = lds.t.pss;
    auto& pmf = lds.t.pmf;
    const int tid = threadIdx.x;
    const int wv = tid >> 6, lane = tid & 63;
    const int rg = wv & 3;           // row group
    const int t256 = tid & 255;      // staging thread within the role
    const int ln = lane & 31, hh = lane >> 5;
    const int n_rows = a.n_q * a.n_rep;
    const BlockPos pos(a, (n_rows + 127) / 128);
    const int h = pos.h, split = pos.split;
    const int row0 = (pos.bx * 4 + rg) * 32;
    const int H_q = a.h_kv * a.n_rep;
    const int r = row0 + ln;
    const bool r_ok = r < n_rows;
    const RowPos rp(a, r_ok ? r : 0);
    const int jq = rp.j, hq = h * a.n_rep + rp.g;
    int nd, u0;
    const int n_blk_tiles = a.block_tiles(pos.bx * 128, min(pos.bx * 128 + 127, n_rows - 1), &nd, &u0);
    const int n_split = a.block_splits(n_blk_tiles);
    if (split >= n_split) return;  // uniform per block
    // The block's tiles go to its splits evenly: blocks go round the XCDs in turn,
    // a split index so often to the same ones, and with splits of `unit` and a
    // short last one half the chip had the long ones (700 queries over 900 tokens,
    // 29 to 50 tiles in two splits: 78.2 us, even 59.6).
    const int per = n_split == a.n_split
                        ? a.by_split.div(n_blk_tiles + n_split - 1)
                        : __builtin_amdgcn_readfirstlane((n_blk_tiles + n_split - 1) / n_split);
    const BlockKeys bk(nd, u0, n_blk_tiles, split, per);
    const bool direct = n_split == 1 && !a.apart;
    const int n_tiles = bk.t_hi - bk.t_lo;
    const int raw_end = a.raw0 + a.n_raw;
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    if (wv < 4) {
        // ================= score wavefront
        const RowKeys vis(a, jq);
        h8 qb[16];
        {
            const __half* qrow = a.q + ((size_t)jq * H_q + hq) * 512;
#pragma unroll
            for (int st = 0; st < 16; st++) {
                const uint4 v = *reinterpret_cast<const uint4*>(qrow + 16 * st + 8 * hh);
                qb[st] = __builtin_bit_cast(h8, r_ok ? v : uint4{0u, 0u, 0u, 0u});
            }
        }
        // K tile staging: thread t -> key t / 8, 64 B at (t % 8) * 32 halves
        const int ld_key = t256 >> 3, ld_off = (t256 & 7) * 32;
        const __half* kg = a.k + (size_t)h * 256 + ld_off;
        uint4 pk[4];
#pragma unroll
        for (int i = 0; i < 4; i++) pk[i] = uint4{0u, 0u, 0u, 0u};
        auto gload = [&](int i0) {  // tile i0 of the split
            const int t = bk.t_lo + i0, b0 = bk.base(t);
            const int key = bk.dec(t) ? b0 + ld_key : min(a.raw0 + b0 + ld_key, raw_end - 1);
            const uint4* ksrc = reinterpret_cast<const uint4*>(kg + (size_t)key * a.h_kv * 256);
#pragma unroll
            for (int i = 0; i < 4; i++) pk[i] = ksrc[i];
        };
        auto lstore = [&](int buf) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                *reinterpret_cast<uint4*>(&ks[buf][ld_key][ld_off + 8 * i]) = pk[i];
        };
        auto kread = [&](int buf, int half, h8 (&kop)[8]) {
#pragma unroll
            for (int i = 0; i < 8; i++)
                kop[i] = *reinterpret_cast<const h8*>(&ks[buf][ln][16 * (8 * half + i) + 8 * hh]);
        };
        if (n_tiles > 0) {
            gload(0);
            lstore(0);
        }
        if (n_tiles > 1) {
            gload(1);
            lstore(1);
        }
        if (n_tiles > 2) gload(2);
        __syncthreads();  // prologue: K tiles 0, 1 and V^T tile 0 staged
        // Weights are rounded to fp16 except a row's reference key's, which is 1.
        // Blocks that run all their keys in one go raise the reference at every
        // new maximum of the first 8 tiles, so a row of few keys (where one
        // weight counts) has its largest one exact; splits have that from their
        // several references.  A layer's pass has fewer of them than one launch
        // per event had, and raises it so too: 200 tokens after 300, 2.86e-4 from
        // float64 without, 2.68e-4 with, 2.72e-4 in a launch per event.
        const int n_eager = n_split == 1 || a.ev_cap > 0 ? 8 : 0;
        const float sc2 = a.sc * LOG2E;  // scores in log2 units: a weight is one exp2
        float m_ref = M_NONE;
        f32x16 s2[2];
        {
            h8 kop[8];
            s2[0] = s2[1] = zero16;
#pragma unroll
            for (int half = 0; half < 2; half++) {
                kread(0, half, kop);
#pragma unroll
                for (int i = 0; i < 8; i++) s2[i & 1] = mfma3232(kop[i], qb[8 * half + i], s2[i & 1]);
            }
        }
        for (int t = 0; t < n_tiles; t++) {
            const int nxt = (t + 1) % NKB;
            float sc[16];
#pragma unroll
            for (int e = 0; e < 16; e++) sc[e] = s2[0][e] + s2[1][e];
            h8 kop[8];
            kread(nxt, 0, kop);
            // ---- S(t + 1), first half, under the scaling, mask and row maximum
            // of tile t; a tile every row of the wavefront sees whole (all but
            // the last few of a block) skips the mask
            float lmax = -INFINITY;
            const uint32_t mask = vis.tile(bk.dec(bk.t_lo + t), bk.base(bk.t_lo + t));
            if (__ballot(mask != ~0u) == 0ull) {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    s2[i & 1] = mfma3232(kop[i], qb[i], i < 2 ? zero16 : s2[i & 1]);
#pragma unroll
                    for (int e = 2 * i; e < 2 * i + 2; e++) {
                        sc[e] *= sc2;
                        lmax = fmaxf(lmax, sc[e]);
                    }
                }
            } else {
                const uint32_t mb = mask >> (4 * hh);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    s2[i & 1] = mfma3232(kop[i], qb[i], i < 2 ? zero16 : s2[i & 1]);
#pragma unroll
                    for (int e = 2 * i; e < 2 * i + 2; e++) {  // key 8 (e / 4) + 4 hh + e % 4
                        sc[e] = (mb >> (8 * (e >> 2) + (e & 3))) & 1u ? sc[e] * sc2 : -INFINITY;
                        lmax = fmaxf(lmax, sc[e]);
                    }
                }
            }
            kread(nxt, 1, kop);
            // ---- raise the row's reference maximum only when needed; the
            // output wavefront rescales its accumulators and sums by fac
            float fac = 1.0f;
            if (__ballot(lmax > m_ref + (t < n_eager ? 0.0f : GAP32)) != 0ull) {
                const float rmax = fmaxf(lmax, __shfl_xor(lmax, 32, 64));
                const float m_new = fmaxf(m_ref, rmax);
                if (m_new > m_ref) {
                    fac = __builtin_amdgcn_exp2f(m_ref - m_new);  // 0 from M_NONE (the sums are still 0)
                    m_ref = m_new;
                }
            }
            // ---- S(t + 1), second half; tile t's scores go to the output side
#pragma unroll
            for (int i = 0; i < 8; i++) s2[i & 1] = mfma3232(kop[i], qb[8 + i], s2[i & 1]);
#pragma unroll
            for (int q4 = 0; q4 < 4; q4++)
                pss[t & 1][rg][q4][lane] = f4{sc[4 * q4], sc[4 * q4 + 1], sc[4 * q4 + 2], sc[4 * q4 + 3]};
            pmf[t & 1][rg][lane] = float2{m_ref, fac};
            // ---- stage K tile t + 2 (its slot last held tile t - 1), load t + 3
            if (t + 2 < n_tiles) {
                lstore((t + 2) % NKB);
                if (t + 3 < n_tiles) gload(t + 3);
            }
            __syncthreads();  // tile t
        }
        __syncthreads();  // the output side's last tile
    } else {
        // ================= output wavefront
        f32x16 acc[8];
#pragma unroll
        for (int t2 = 0; t2 < 8; t2++) acc[t2] = zero16;
        // V^T tile staging: thread t -> dim t, the tile's 32 keys (64 B)
        const __half* vg = a.vt + ((size_t)h * 256 + t256) * a.ld_vt;
        uint4 pv[4];
#pragma unroll
        for (int i = 0; i < 4; i++) pv[i] = uint4{0u, 0u, 0u, 0u};
        auto gload = [&](int i0) {
            const int t = bk.t_lo + i0;
            const uint4* vsrc =
                reinterpret_cast<const uint4*>(vg + (bk.dec(t) ? 0 : a.raw0) + bk.base(t));
#pragma unroll
            for (int i = 0; i < 4; i++) pv[i] = vsrc[i];
        };
        auto vmask = [](uint32_t w, int i, int nv) {
            return 2 * i + 1 < nv ? w : (2 * i < nv ? (w & 0xFFFFu) : 0u);
        };
        auto lstore = [&](int buf, int i0) {
            const int t = bk.t_lo + i0;
            const int nv = bk.dec(t) ? KT : a.n_raw - bk.base(t);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                *reinterpret_cast<uint2*>(&vs[buf][t256][8 * i]) = uint2{pv[i].x, pv[i].y};
                *reinterpret_cast<uint2*>(&vs[buf][t256][8 * i + 4]) = uint2{pv[i].z, pv[i].w};
            }
            if (nv < KT) {  // the last raw tile: V^T columns past its keys cleared
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint4 v = pv[i];
                    *reinterpret_cast<uint2*>(&vs[buf][t256][8 * i]) =
                        uint2{vmask(v.x, 4 * i, nv), vmask(v.y, 4 * i + 1, nv)};
                    *reinterpret_cast<uint2*>(&vs[buf][t256][8 * i + 4]) =
                        uint2{vmask(v.z, 4 * i + 2, nv), vmask(v.w, 4 * i + 3, nv)};
                }
            }
        };
        // O^T += V^T P^T for tile u: 8 tiles of 32 dims x 2 K-steps of 16 keys
        float l_part = 0.0f, m_last = M_NONE;
        auto pv_tile = [&](int u) {
            const int cur = u % NKB;
            // the tile's V^T operands first: their LDS latency runs under the
            // exponentials below
            h8 vop[2][8];
#pragma unroll
            for (int sp = 0; sp < 2; sp++)
#pragma unroll
                for (int t2 = 0; t2 < 8; t2++) {
                    const uint2 va = *reinterpret_cast<const uint2*>(&vs[cur][32 * t2 + ln][16 * sp + 4 * hh]);
                    const uint2 vb = *reinterpret_cast<const uint2*>(&vs[cur][32 * t2 + ln][16 * sp + 8 + 4 * hh]);
                    vop[sp][t2] = __builtin_bit_cast(h8, uint4{va.x, va.y, vb.x, vb.y});
                }
            const float2 mf = pmf[u & 1][rg][lane];
            const f4 s0 = pss[u & 1][rg][0][lane], s1 = pss[u & 1][rg][1][lane];
            const f4 s2v = pss[u & 1][rg][2][lane], s3 = pss[u & 1][rg][3][lane];
            const float sc[16] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3],
                                  s2v[0], s2v[1], s2v[2], s2v[3], s3[0], s3[1], s3[2], s3[3]};
            m_last = mf.x;
            if (__ballot(mf.y != 1.0f) != 0ull) {
#pragma unroll
                for (int t2 = 0; t2 < 8; t2++) acc[t2] *= mf.y;
                l_part *= mf.y;
            }
            float p[16];
#pragma unroll
            for (int e = 0; e < 16; e++) p[e] = __builtin_amdgcn_exp2f(sc[e] - mf.x);  // 0 where masked
            uint32_t pw[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                pw[e] = pk_rne(p[2 * e], p[2 * e + 1]);
                l_part = add_pair(pw[e], l_part);
            }
            h8 pbv[2];
#pragma unroll
            for (int sp = 0; sp < 2; sp++)
                pbv[sp] = __builtin_bit_cast(h8, uint4{pw[4 * sp], pw[4 * sp + 1], pw[4 * sp + 2], pw[4 * sp + 3]});
#pragma unroll
            for (int sp = 0; sp < 2; sp++)
#pragma unroll
                for (int t2 = 0; t2 < 8; t2++) acc[t2] = mfma3232(vop[sp][t2], pbv[sp], acc[t2]);
        };
        if (n_tiles > 0) {
            gload(0);
            lstore(0, 0);
        }
        if (n_tiles > 1) gload(1);
        __syncthreads();  // prologue
        for (int t = 0; t < n_tiles; t++) {
            if (t >= 1) pv_tile(t - 1);
            // ---- stage V^T tile t + 1 (its slot last held tile t - 2), load t + 2
            if (t + 1 < n_tiles) {
                lstore((t + 1) % NKB, t + 1);
                if (t + 2 < n_tiles) gload(t + 2);
            }
            __syncthreads();  // tile t
        }
        if (n_tiles > 0) pv_tile(n_tiles - 1);
        __syncthreads();  // last tile applied
        const float l_row = l_part + __shfl_xor(l_part, 32, 64);
        // ---- row ln: the output, or its partial triple (dims 32 t + 8 j + 4 hh + c)
        const bool empty = m_last == M_NONE;
        const float f = empty ? 0.0f : (direct ? 1.0f / (l_row + a.eps) : 1.0f);
#pragma unroll
        for (int t2 = 0; t2 < 8; t2++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                *reinterpret_cast<f4*>(&lds.out[rg][ln][32 * t2 + 8 * j + 4 * hh]) =
                    f4{acc[t2][4 * j], acc[t2][4 * j + 1], acc[t2][4 * j + 2], acc[t2][4 * j + 3]} * f;
        wave_sync();
        if (!direct)
            store_rows<32>(a, &lds.out[rg][0][0], __builtin_amdgcn_readfirstlane(row0), h, split, false,
                           empty ? -1e20f : m_last * LN2, empty ? 0.0f : l_row, lane);
    }
    if (direct) {  // uniform per block; gates and stores: half a row group each wavefront
        __syncthreads();
        const int half = tid < 256 ? 0 : 16;
        store_rows<16>(a, &lds.out[rg][half][0], __builtin_amdgcn_readfirstlane(row0 + half), h, split, true,
                       0.0f, 0.0f, lane);
    }
}

// Merge of the key splits, normalisation and gate: one wavefront per (query,
// head) row of a block that was split (the others' rows are written already),
// lane l owning dims 4 l .. 4 l + 3; lane s < n_split holds split s's (m, l)
// pair.  Each group of up to 16 splits has every load in flight before the
// first is used (the first group's with the (m, l) loads, ahead of the
// maximum); the sums run in split order.
constexpr int MG = 16;  // splits per load group
struct MergeArgs {
    const float* part;
    const __half* q;
    __half* out;
    int n_rows, n_split, nb;  // rows, triples a row, merging blocks
    float eps;
    int h_kv, n_rep;  // row order of the wide form: heads in turn, or 1 and H_q
    FastDiv by_kv, by_rep;
};
__device__ __forceinline__ void merge_row(const MergeArgs& p, int row, int n_split) {
    const int lane = threadIdx.x & 63;
    const float* base = p.part + (size_t)row * p.n_split * 258;
    float2 a[MG][2];
    auto load_group = [&](int s0) {
#pragma unroll
        for (int j = 0; j < MG; j++)
            if (s0 + j < n_split) {
                const float* pp = base + (size_t)(s0 + j) * 258 + 4 * lane;
                a[j][0] = *reinterpret_cast<const float2*>(pp);
                a[j][1] = *reinterpret_cast<const float2*>(pp + 2);
            }
    };
    load_group(0);  // in flight with the (m, l) pairs below
    float m = -1e30f, l = 0.0f;
    if (lane < n_split) {
        const float2 ml = *reinterpret_cast<const float2*>(base + (size_t)lane * 258 + 256);
        m = ml.x;
        l = ml.y;
    }
    float M = m;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
    const float w = lane < n_split ? __expf(m - M) : 0.0f;
    const float lw = l * w;
    float num[4] = {0.f, 0.f, 0.f, 0.f}, den = 0.0f;
    for (int s0 = 0; s0 < n_split; s0 += MG) {
        if (s0 > 0) load_group(s0);
#pragma unroll
        for (int j = 0; j < MG; j++)
            if (s0 + j < n_split) {
                const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), s0 + j));
                num[0] = fmaf(a[j][0].x, ws, num[0]);
                num[1] = fmaf(a[j][0].y, ws, num[1]);
                num[2] = fmaf(a[j][1].x, ws, num[2]);
                num[3] = fmaf(a[j][1].y, ws, num[3]);
                den += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lw), s0 + j));
            }
    }
    const uint2 gw = *reinterpret_cast<const uint2*>(p.q + (size_t)row * 512 + 256 + 4 * lane);
    const h4 g = __builtin_bit_cast(h4, gw);
    float o[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
        o[c] = num[c] / (den + p.eps) * (1.0f / (1.0f + expf(-(float)g[c])));
    *reinterpret_cast<uint2*>(p.out + (size_t)row * 256 + 4 * lane) =
        uint2{pk_rne(o[0], o[1]), pk_rne(o[2], o[3])};
}

// Blocks [0, nb_m): rows 4 b .. + 3, one wavefront each; the rest copy new
// tokens to the ring, 8 bytes a thread and tensor.
__device__ __forceinline__ void ring_pieces(const RingArgs& g, int b) {
    const int i = b * 256 + threadIdx.x, t = g.by_token.div(i);
    if (t >= g.n) return;
    const int per = g.h_kv * 64, e = (i - t * per) * 4;  // pieces per token
    int slot = g.slot0 + t;
    slot = slot >= g.ring_cap ? slot - g.ring_cap : slot;
    const size_t src = (size_t)t * per * 4 + e, dst = (size_t)slot * per * 4 + e;
    *reinterpret_cast<uint2*>(g.ring_k + dst) = *reinterpret_cast<const uint2*>(g.src_k + src);
    *reinterpret_cast<uint2*>(g.ring_v + dst) = *reinterpret_cast<const uint2*>(g.src_v + src);
    *reinterpret_cast<uint2*>(g.ring_u + dst) = *reinterpret_cast<const uint2*>(g.src_u + src);
}
// A block for a row of many splits: each wavefront sums a quarter of them, every
// load and the gate in flight, and the four meet in LDS.  One wavefront takes 64
// splits in four round trips and the gate in a fifth: 120 rows 8.3 us, 504 rows
// 9.1; this way 4.3 and 6.8.  With 8 KV heads blocks take them in turn, as the
// 16-row kernel's blocks do, and a row is merged on the XCD whose L2 holds its
// triples (16 queries of 32 / 8 heads over 900 tokens: 12.7 us, 17.4 row by row; of
// 24 / 4 heads 15.1, 14.5 row by row).
__device__ __forceinline__ void merge_row_wide(const MergeArgs& p, int row) {
    __shared__ __align__(16) float s_num[4][256];
    __shared__ float s_den[4];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const float* base = p.part + (size_t)row * p.n_split * 258;
    const int per = (p.n_split + 3) / 4, lo = wv * per, n = min(per, p.n_split - lo);  // per <= MG
    float2 a[MG][2];
#pragma unroll
    for (int j = 0; j < MG; j++)
        if (j < n) {
            const float* pp = base + (size_t)(lo + j) * 258 + 4 * lane;
            a[j][0] = *reinterpret_cast<const float2*>(pp);
            a[j][1] = *reinterpret_cast<const float2*>(pp + 2);
        }
    const float2 ml = *reinterpret_cast<const float2*>(base + (size_t)min(lane, p.n_split - 1) * 258 + 256);
    const float gate = __half2float(p.q[(size_t)row * 512 + 256 + threadIdx.x]);
    float M = ml.x;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
    const float w = __expf(ml.x - M), lw = ml.y * w;  // lanes past the splits repeat the last
    float num[4] = {0.f, 0.f, 0.f, 0.f}, den = 0.0f;
#pragma unroll
    for (int j = 0; j < MG; j++)
        if (j < n) {
            const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), lo + j));
            num[0] = fmaf(a[j][0].x, ws, num[0]);
            num[1] = fmaf(a[j][0].y, ws, num[1]);
            num[2] = fmaf(a[j][1].x, ws, num[2]);
            num[3] = fmaf(a[j][1].y, ws, num[3]);
            den += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lw), lo + j));
        }
    *reinterpret_cast<float4*>(&s_num[wv][4 * lane]) = make_float4(num[0], num[1], num[2], num[3]);
    if (lane == 0) s_den[wv] = den;
    __syncthreads();
    const int t = threadIdx.x;
    const float v = (s_num[0][t] + s_num[1][t]) + (s_num[2][t] + s_num[3][t]);
    const float d = (s_den[0] + s_den[1]) + (s_den[2] + s_den[3]);
    p.out[(size_t)row * 256 + t] = __float2half(v / (d + p.eps) * (1.0f / (1.0f + expf(-gate))));
}
__global__ __launch_bounds__(256) void prefill_finish_wide_kernel(MergeArgs m, RingArgs g) {
    const int b = blockIdx.x;
    if (b >= m.nb) {
        ring_pieces(g, b - m.nb);
        return;
    }
    const int r = m.by_kv.div(b), h = b - r * m.h_kv;  // row of the KV head
    const int j = m.by_rep.div(r);
    merge_row_wide(m, j * m.h_kv * m.n_rep + h * m.n_rep + r - j * m.n_rep);
}
__global__ __launch_bounds__(256) void prefill_finish_kernel(MergeArgs m, RingArgs g) {
    const int b = blockIdx.x;
    if (b >= m.nb) {
        ring_pieces(g, b - m.nb);
        return;
    }
    const int row = b * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row < m.n_rows) merge_row(m, row, m.n_split);  // uniform per wavefront
}
// Blocks of unlike split counts, those of one split written out already:
// block_rows (a power of two) rows of a KV head each.
__global__ __launch_bounds__(256) void prefill_finish_ragged_kernel(MergeArgs m, RingArgs g, PrefillArgs a,
                                                                    int block_rows) {
    const int b = blockIdx.x;
    if (b >= m.nb) {
        ring_pieces(g, b - m.nb);
        return;
    }
    const int row = b * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row >= m.n_rows) return;
    const int j = a.by_hq.div(row), hq = row - j * a.h_kv * a.n_rep;
    const int first = (j * a.n_rep + RowPos(a, hq).g) & -block_rows;
    int nd, u0;
    const int ns = a.block_splits(
        a.block_tiles(first, min(first + block_rows, a.n_q * a.n_rep) - 1, &nd, &u0));
    if (ns > 1 || a.apart) merge_row(m, row, ns);
}

}  // namespace pf

namespace {
// RoPE frequencies by the host's powf, as the attention kernels' table has them
// (four powf a lane on the GPU were more than a row's decode).
DecompArgs with_rope(DecompArgs a) {
    thread_local float last_base = NAN;  // unlike every base
    thread_local float freq[32];
    if (a.rope_base != last_base) {
        for (int i = 0; i < 32; i++) freq[i] = powf(a.rope_base, -2.0f * (float)i / 64.0f);
        last_base = a.rope_base;
    }
    memcpy(a.freq, freq, sizeof(freq));
    return a;
}
int gather_blocks(const GatherArgs& g) { return g.n > 0 ? (g.n + 31) / 32 * g.h_kv : 0; }
bool long_decode(const DecompArgs& a) {
    // 4 KV heads, 4 / 16 tokens a block: 1,024 tokens 11.3 / 12.6 us, 2,000
    // 15.9 / 15.8, 8,192 39.6 / 37.0, 32,640 153 / 121
    return a.n_tok / pf::TB_LONG * a.h_kv >= 2 * device_cu_count();
}
}  // namespace

hipError_t launch_prefill_finish(const PrefillArgs& a, const RingArgs* ring, hipStream_t st) {
    const int n_rows = a.n_q * a.h_kv * a.n_rep;
    // (wide at up to 16 splits: 1 query over 200 tokens 8.0 -> 7.7 us, 48 over 900, 1,152
    // rows of 15 splits, 22.2 -> 21.2; 6,144 rows of 5 splits the other way, 48.5 -> 50.3)
    const bool wide = a.uniform && (a.n_split > pf::MG ||
                                    (a.n_split > 4 && n_rows <= 8 * device_cu_count()));
    const bool turn = a.h_kv % 8 == 0;  // XCDs
    const pf::MergeArgs m{a.part, a.q, a.out, n_rows, a.n_split,
                          wide ? n_rows : a.n_split > 1 || a.apart ? (n_rows + 3) / 4 : 0, a.eps,
                          turn ? a.h_kv : 1, turn ? a.n_rep : a.h_kv * a.n_rep,
                          turn ? a.by_kv : FastDiv(1), turn ? a.by_rep : a.by_hq};
    RingArgs g = ring ? *ring : RingArgs{};
    g.by_token = FastDiv(std::max(1, g.h_kv * 64));
    const dim3 grid(m.nb + (g.n * g.h_kv * 64 + 255) / 256);
    if (grid.x == 0) return hipSuccess;
    if (wide)
        hipLaunchKernelGGL(pf::prefill_finish_wide_kernel, grid, dim3(256), 0, st, m, g);
    else if (a.uniform)
        hipLaunchKernelGGL(pf::prefill_finish_kernel, grid, dim3(256), 0, st, m, g);
    else
        hipLaunchKernelGGL(pf::prefill_finish_ragged_kernel, grid, dim3(256), 0, st, m, g, a,
                           prefill_block_rows(a.n_q * a.n_rep));
    return hipGetLastError();
}

hipError_t launch_decompress(const DecompArgs& args, hipStream_t st) {
    if (args.n_tok <= 0) return hipSuccess;
    const DecompArgs a = with_rope(args);
    if (long_decode(a))
        hipLaunchKernelGGL(pf::decompress_kernel<pf::TB_LONG>,
                           dim3((a.n_tok + pf::TB_LONG - 1) / pf::TB_LONG, a.h_kv),
                           dim3(pf::BLK_THR), 0, st, a);
    else
        hipLaunchKernelGGL(pf::decompress_kernel<4>, dim3((a.n_tok + 3) / 4, a.h_kv),
                           dim3(pf::BLK_THR), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_decompress_gather(const DecompArgs& args, const GatherArgs& g, hipStream_t st) {
    if (args.n_tok <= 0) return launch_ring_gather(g, st);
    if (g.n <= 0) return launch_decompress(args, st);
    const DecompArgs d = with_rope(args);
    const int tb = long_decode(d) ? pf::TB_LONG : 4, nx_d = (d.n_tok + tb - 1) / tb;
    const dim3 grid(nx_d * d.h_kv + gather_blocks(g));
    if (tb == 4)
        hipLaunchKernelGGL(pf::decompress_gather_kernel<4>, grid, dim3(pf::BLK_THR), 0, st, d, g, nx_d);
    else
        hipLaunchKernelGGL(pf::decompress_gather_kernel<pf::TB_LONG>, grid, dim3(pf::BLK_THR), 0, st,
                           d, g, nx_d);
    return hipGetLastError();
}

hipError_t launch_compress_decode(const CompressJob& k, const CompressJob& v, const DecompArgs& args,
                                  const GatherArgs& g, hipStream_t st) {
    const DecompArgs d = with_rope(args);
    // the decode covers exactly the compressed rows: token t, KV head h is row t h_kv + h
    if (k.n != v.n || d.n_tok * d.h_kv != k.n || d.tok0 != d.key0 || d.start_pos != 0)
        return hipErrorInvalidValue;
    const int nb_k = (k.n + 3) / 4;
    hipLaunchKernelGGL(pf::compress_decode_kernel, dim3(v.n + nb_k + gather_blocks(g)),
                       dim3(pf::BLK_THR), 0, st, k, v, d, g, nb_k);
    return hipGetLastError();
}

hipError_t launch_compress_gather(const CompressJob& k, const CompressJob& v, const GatherArgs& g,
                                  hipStream_t st) {
    const int k_many = compress_k_many(k.n);
    const int nb_k = k_many ? (k.n + 4 * KR - 1) / (4 * KR) : (k.n + 3) / 4;
    const int nb_v = (v.n + VR - 1) / VR;
    hipLaunchKernelGGL(pf::compress_gather_kernel, dim3(nb_k + nb_v + gather_blocks(g)),
                       dim3(pf::BLK_THR), 0, st, k, v, g, nb_k, nb_v, k_many);
    return hipGetLastError();
}

hipError_t launch_ring_gather(const GatherArgs& a, hipStream_t st) {
    if (a.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(pf::ring_gather_kernel, dim3(gather_blocks(a)), dim3(pf::BLK_THR), 0, st, a);
    return hipGetLastError();
}

namespace {
// Few query rows (a handful of queries): the 16-row kernel, two blocks per CU
// (more, shorter splits); many: the role-specialised 32-row kernel (half the
// LDS operand traffic per flop).
bool few_rows(int n_rows) { return n_rows <= 128; }
}  // namespace

int prefill_block_rows(int n_rows) { return few_rows(n_rows) ? 64 : 128; }

void prefill_plan(PrefillArgs& a, size_t max_bytes) {
    // Blocks that run at once: 2 per CU for the 16-row kernel (72 KB of LDS
    // each), 1 for the 32-row kernel (142 KB).
    const int n_rows = a.n_q * a.n_rep, br = prefill_block_rows(n_rows);
    const int nb = (n_rows + br - 1) / br;
    const bool few = few_rows(n_rows);
    const int slots = (few ? 2 : 1) * device_cu_count();
    a.by_rep = FastDiv(a.n_rep);
    a.by_hq = FastDiv(a.h_kv * a.n_rep);
    a.by_kv = FastDiv(a.h_kv);
    auto tiles_of = [&](int b) {
        int nd, u0;
        return a.block_tiles(b * br, std::min(b * br + br, n_rows) - 1, &nd, &u0);
    };
    int t_max = 1, t_min = 1 << 30;
    for (int b = 0; b < nb; b++) {
        const int t = tiles_of(b);
        t_max = std::max(t_max, t);
        t_min = std::min(t_min, t);
    }
    // Where the shortest block would have three quarters of the splits and there
    // is room, it gets as many as the others, and the merge does not work out each
    // row's count (128 queries of 8 / 1 heads over 900 tokens, 15 to 17 splits: 25.3
    // us, 21.7 in 17).
    auto set_splits = [&](int k) {
        a.unit = (t_max + k - 1) / k;
        a.n_split = (t_max + a.unit - 1) / a.unit;
        a.by_unit = FastDiv(a.unit);
        a.round_up = a.unit - 1;
        const int least = a.block_splits(t_min);
        a.uniform = few || least == a.n_split ||
                    (4 * least >= 3 * a.n_split && nb * a.h_kv * a.n_split <= slots);
        if (a.uniform) {  // the same quotient for all
            a.by_unit = FastDiv(1u << 20);
            a.round_up = a.n_split << 20;
        }
    };
    // At least as many splits as one round holds: a weight is rounded to fp16
    // but for its tile's largest where that sets the reference (a split's first
    // tile), so short splits lose less.  16 queries over 900 tokens, whatever is
    // faster (10 splits): 2.80e-4 from float64, 29 splits of a tile 2.53e-4, the
    // output's own rounding being 2.07e-4.
    int k_min = std::max(1, std::min({64, t_max, slots / (nb * a.h_kv)}));
    while (k_min > 1 && a.triple_bytes(k_min) > max_bytes) k_min--;
    int best_k = k_min;
    if (few) {
        a.apart = true;  // gating 16 rows in turn in the block takes longer than the finishing launch
    } else {
        // More where it is faster.  With splits of at most `unit` tiles, the
        // launch takes, in tiles of time:
        //   one round of the longest block when they all fit at once;
        //   else the work over the slots plus half a block of tail (they start
        //   longest first), or whole rounds when the blocks are equally long (a
        //   few blocks past a round cost a whole round); the fullest engine's work
        //   where they split unlike and are few.
        // A block costs about 4 tiles beside its own (entry, first loads, output);
        // splitting costs the finishing launch, about 4, and 0.045 a block for its
        // triples (128 rows x 1 KB written and read).  Where one round holds every
        // block, gating the rows inside it (a.apart = false) is not free either: a
        // wavefront gates up to 16 rows in turn, 0.29 each, with nothing else on its
        // CU.
        const bool even = t_max - t_min <= t_max / 8;
        // Blocks go to the shader engines (8 CUs) in turn: where they split unlike,
        // the fullest engine counts, with every fourth or eighth index in use or
        // fewer (400 queries of a prompt, 160 blocks in up to 4 splits: two rounds,
        // 33.6 us; 140 in up to 3: 26.3), and the last eighth of the slots is not
        // filled in one round (550 over 100 tokens: 228 blocks 36.7 us, 164 32.5).
        const int engines = std::min(64, std::max(1, slots / 8));
        auto engine_time = [&](int units) {
            int most = 0, n[64] = {};
            float load = 0.0f, w[64] = {};
            for (int b = 0, i = 0; b < nb; b++) {
                const int t = tiles_of(nb - 1 - b), s = a.block_splits(t), per = (t + s - 1) / s;
                for (int h = 0; h < a.h_kv; h++, i += a.n_split)
                    for (int e = i; e < i + s; e++) {
                        most = std::max(most, ++n[e % engines]);
                        load = std::max(load, w[e % engines] += per + 4);
                    }
            }
            return most <= 8 && units <= slots - slots / 8 ? a.unit + 4.0f : load / 8 + 0.5f * a.unit;
        };
        const float gate = 0.29f * std::min(16, n_rows);
        const int step = std::max(1, nb / 64);  // enough blocks to add up
        float best = 0.0f;
        for (int k = k_min; k <= std::min(64, t_max); k++) {
            set_splits(k);
            // (the workspace stays: past 256 MB a finer tail is not worth it)
            if (k > k_min && a.triple_bytes(k) > std::min(max_bytes, (size_t)256 << 20)) break;
            float units = 0.0f, tiles = 0.0f;
            for (int b = 0; b < nb; b += step) {
                const int t = tiles_of(b);
                const float w = (float)std::min(step, nb - b) * a.h_kv;
                units += w * a.block_splits(t);
                tiles += w * t;
            }
            const float least = (tiles + 4 * units) / slots;
            if (k > k_min && least + 4.0f + 0.045f * units >= best) break;  // and so any finer
            const float rounds = std::ceil(units / slots);
            float est = a.uniform && (rounds <= 1.0f || even) ? rounds * (a.unit + 4)
                        : a.uniform || rounds > 4.0f          ? least + 0.5f * a.unit
                                                              : engine_time((int)units);
            bool apart = !a.out;
            if (k > 1 || (rounds <= 1.0f && gate > 4.0f + 0.045f * units && a.triple_bytes(1) <= max_bytes)) {
                est += 4.0f + 0.045f * units;
                apart |= rounds <= 1.0f;
            } else if (rounds <= 1.0f) {
                est += gate;
            }
            if (k == k_min || est < best) {
                best = est;
                best_k = k;
                a.apart = apart;
            }
        }
    }
    set_splits(best_k);
    a.by_split = FastDiv(a.n_split);
}

hipError_t launch_prefill_attn(const PrefillArgs& a, hipStream_t st) {
    const int n_rows = a.n_q * a.n_rep, br = prefill_block_rows(n_rows), nb = (n_rows + br - 1) / br;
    if (few_rows(n_rows)) {
        pf::FewBlocks f{};
        for (int b = 0; b < nb; b++)
            f.n[b] = a.block_tiles(b * br, std::min(b * br + br, n_rows) - 1, &f.nd[b], &f.u0[b]);
        hipLaunchKernelGGL(pf::prefill_attn_kernel, dim3(nb, a.h_kv, a.n_split), dim3(256), 0, st, a, f);
    } else {
        hipLaunchKernelGGL(pf::prefill_attn_rs_kernel, dim3((unsigned)nb * a.h_kv * a.n_split), dim3(512), 0,
                           st, a);
    }
    return hipGetLastError();
}

}  // namespace khq
