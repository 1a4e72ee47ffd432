// Attention with one sequence's keys over many workgroups, for decoding at long
// contexts and in small batches and for short chunks at long contexts,
// bit-equal to the block walk of kernels/attention_gqa.h:404-547 /
// ref_qwen3.py:210-266.
//
// k_attn_decode.hip gives a sequence one workgroup per head (or per KV head),
// which walks the key blocks chunk by chunk: a 4000-key context is six serial
// chunks of ~6 us on 16 of 256 CUs.  Of the recurrence only the den/res chain
// is sequential, and it is two operations per block and dimension; everything
// else needs a block and the running maximum, a prefix max of the block
// maxima.  So three launches, each over every (sequence, KV head, 4 blocks):
//   score  one wave per block: S = q8.k8^T of the KV head's two query heads,
//          s and the block maxima to the workspace; its prologue is the head
//          epilogue of the new token's projection rows (Q, K: RMSNorm, RoPE,
//          quant; V: quant), the workgroup of the last block writing the page
//          slot
//   pv     one wave per block: nmm_j = max of the block maxima 0..j, P =
//          exp(s - nmm_j), psum_j, P8, pv_j = f32(P8.V) * pmax_j to the
//          workspace
//   chain  one workgroup per (sequence, head): corr_j = exp(nmm_{j-1} -
//          nmm_j), den = den * corr_j + psum_j, res = res * corr_j + pv_j in
//          block order, then the output quantisation
// with the reference's rounding points.  At 4000 keys and b = 1 the launches
// take 4.5, 5.0 and 7.1 us (the fused launch they replace, with its down and
// Q|K|V projections: 43.6), at 24 rows x 2048 keys 14.8, 15.5 and 6.3 us;
// score and pv are bound by latency below ~1000 blocks, then by the K and V
// stream (3.4 TB/s), chain by the walk over the blocks (one per ~30 cycles).
// Two or four blocks per wave were slower at every size (24 x 2048: 1998 us a
// step against 2109 and 2268), and so was prefetching the next GEMVs' weights
// beside pv and chain (4000 keys: 953 against 1025 us a token).
// The kernel boundaries are the only
// synchronisation.  pv_j is 512 bytes per head and block, half of what the
// block's K and V rows hold for the two heads, so the split pays while the
// launch is short of workgroups, not when a batch fills the chip
// (attn_split_batch).
#include "q3_attn_v.h"
#include "q3_device.h"
#include "q3_epi.h"
#include "q3_kernels.h"

namespace q3 {
namespace {

constexpr int kWaves = 4;   // blocks per workgroup (one per wave)
constexpr int kGrp = 2;     // query heads per KV head
constexpr float kFloor = -3.402823466e38f;  // the walk's first maximum (attention_gqa.h:418)

struct Unit {
  int row, split, kvh, nblk;
  uint32_t kv_len;
  const uint16_t *table;
};

// Workgroup id -> (KV head, sequence, 4-block run): ids with equal residues
// mod 8 run on one XCD, so the KV heads of a run (which share its page-table
// and scale lines) get ids with one residue.
__device__ __forceinline__ Unit make_unit(const SplitArgs &a) {
  const int id = static_cast<int>(blockIdx.x);
  const int t = id >> 3;
  const int u = (t / a.kv_heads) * 8 + (id & 7);
  Unit w;
  w.kvh = t % a.kv_heads;
  w.row = u % a.rows;
  w.split = u / a.rows;
  w.kv_len = a.row_pos ? static_cast<uint32_t>(a.row_pos[w.row]) + 1 : a.kv_len;
  w.nblk = static_cast<int>((w.kv_len + 31) / 32);
  w.table = a.row_pos ? a.table + static_cast<int64_t>(w.row) * a.ld_table : a.table;
  return w;
}

__global__ void __launch_bounds__(kWaves * 64) split_score_kernel(SplitArgs a) {
  __shared__ __align__(16) int8_t q8s[kGrp][HD];
  __shared__ __align__(16) int8_t knew[HD];
  __shared__ float qss[kGrp], ksnew;
  const Unit u = make_unit(a);
  if (u.split * kWaves >= u.nblk) return;
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int blk = u.split * kWaves + wave;
  const int jb = min(blk, u.nblk - 1);
  const int j = jb * 32;
  const int pos0 = static_cast<int>(u.kv_len) - 1;
  const bool tail = (u.split + 1) * kWaves >= u.nblk;  // holds the new token's block
  // this wave's projection row: waves 0, 1 a query head each, 2 K, 3 V
  const int qh = u.kvh * kGrp + (wave & 1);
  const float *src = wave < kGrp  ? a.fq + static_cast<int64_t>(u.row) * a.ldq + qh * HD
                     : wave == 2 ? a.fk + static_cast<int64_t>(u.row) * a.ldk + u.kvh * HD
                                 : a.fv + static_cast<int64_t>(u.row) * a.ldk + u.kvh * HD;
  float t0 = src[lane], t1 = src[lane + 64];
  const float *nw = wave < kGrp ? a.nq : a.nk;
  const float w0 = nw[lane], w1 = nw[lane + 64];
  const float c = a.cos_t[static_cast<int64_t>(pos0) * 64 + lane];
  const float sn = a.sin_t[static_cast<int64_t>(pos0) * 64 + lane];
  // K rows and scales of the wave's block (keys past the last repeat it)
  const uint32_t page = u.table[static_cast<uint32_t>(j) / a.page_tokens];
  const uint32_t slot0 = static_cast<uint32_t>(j) % a.page_tokens;
  const int8_t *kb = a.k + page * a.page_bytes + slot0 * a.row_bytes + u.kvh * HD;
  const int8_t *ksb = reinterpret_cast<const int8_t *>(a.ks) + page * a.scale_page_bytes + slot0 * a.scale_row_bytes;
  const int last = pos0 - j;
  const int kg = lane >> 3, kb16 = 16 * (lane & 7);
  const int kcl = 8 * ((lane >> 1) & 3) + kg;  // key whose score the lane ends with
  int4 kw[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    kw[e] = *reinterpret_cast<const int4 *>(kb + min(8 * e + kg, last) * a.row_bytes + kb16);
  float kscale = reinterpret_cast<const float *>(ksb + min(kcl, last) * a.scale_row_bytes)[u.kvh];
  uint32_t npage = 0;
  if (tail) npage = u.table[static_cast<uint32_t>(pos0) / a.page_tokens];
  // ---- head epilogues (norm_rope_quant.h:17-86, group_gemm.h:173-193) ----
  if (wave < kGrp || tail) {
    if (wave != 3) head_norm_rope_regs(t0, t1, w0, w1, c, sn, a.inv_hd, true);
    const float scale = __fmul_rn(max64(fmaxf(fabsf(t0), fabsf(t1))), inv127());
    const int8_t q0 = static_cast<int8_t>(quant1(t0, scale));
    const int8_t q1 = static_cast<int8_t>(quant1(t1, scale));
    if (wave < kGrp) {
      q8s[wave][lane] = q0;
      q8s[wave][lane + 64] = q1;
      if (lane == 0) qss[wave] = scale;
      if (tail) {  // the int8 row for the record
        int8_t *row8 = a.q8 + static_cast<int64_t>(u.row) * a.ldq8 + qh * HD;
        row8[lane] = q0;
        row8[lane + 64] = q1;
        if (lane == 0) a.qs[static_cast<int64_t>(u.row) * a.ldqs + qh] = scale;
      }
    } else {
      if (wave == 2) {
        knew[lane] = q0;
        knew[lane + 64] = q1;
        if (lane == 0) ksnew = scale;
      }
      const uint32_t slot = static_cast<uint32_t>(pos0) % a.page_tokens;
      int8_t *row8 = (wave == 2 ? a.k : a.v) + npage * a.page_bytes + slot * a.row_bytes + u.kvh * HD;
      float *sp = reinterpret_cast<float *>(reinterpret_cast<int8_t *>(wave == 2 ? a.ks : a.vs) +
                                            npage * a.scale_page_bytes + slot * a.scale_row_bytes) + u.kvh;
      row8[lane] = q0;
      row8[lane + 64] = q1;
      if (lane == 0) *sp = scale;
    }
  }
  __syncthreads();
  if (blk >= u.nblk) return;
  if (pos0 < j + 32) {  // the new token's K row from LDS (its page slot may not be visible)
    const int4 kn = *reinterpret_cast<const int4 *>(knew + kb16);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (j + 8 * e + kg >= pos0) kw[e] = kn;
    if (j + kcl >= pos0) kscale = ksnew;
  }
  const int64_t ws0 = (static_cast<int64_t>(u.row) * a.heads + u.kvh * kGrp) * a.ldb + jb;
#pragma unroll
  for (int h = 0; h < kGrp; ++h) {
    const int4 q = *reinterpret_cast<const int4 *>(q8s[h] + kb16);
    int p[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p[e] = sdot4(q.x, kw[e].x, 0);
      p[e] = sdot4(q.y, kw[e].y, p[e]);
      p[e] = sdot4(q.z, kw[e].z, p[e]);
      p[e] = sdot4(q.w, kw[e].w, p[e]);
    }
    // exact int32 sums over the 8 lanes of a key, scattered over lane bits
    // 2, 1, 0 so that lanes 2m, 2m + 1 end with key kcl
    const bool b2 = lane & 4, b1 = lane & 2;
    int k0 = b2 ? p[2] : p[0], k1 = b2 ? p[3] : p[1];
    k0 += lane_xor<4>(b2 ? p[0] : p[2]);
    k1 += lane_xor<4>(b2 ? p[1] : p[3]);
    int acc = b1 ? k1 : k0;
    acc += lane_xor<2>(b1 ? k0 : k1);
    acc += lane_xor<1>(acc);
    float s = -INFINITY;
    if (j + kcl <= pos0) {
      s = __fmul_rn(static_cast<float>(acc), kscale);
      s = __fmul_rn(s, qss[h]);
      s = __fmul_rn(s, a.qk_scale);
    }
    const float bm = max64(s);
    const int64_t wb = ws0 + h * a.ldb;
    if ((lane & 1) == 0) a.ws_s[wb * 32 + kcl] = s;
    if (lane == 0) a.ws_bmax[wb] = bm;
  }
}

__global__ void __launch_bounds__(kWaves * 64) split_pv_kernel(SplitArgs a) {
  __shared__ uint64_t tab[32];
  __shared__ __align__(16) int8_t vst[kWaves][32 * HD];
  __shared__ __align__(16) int8_t p8s[kWaves][kGrp][32];
  const Unit u = make_unit(a);
  if (u.split * kWaves >= u.nblk) return;
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int blk = u.split * kWaves + wave;
  const int jb = min(blk, u.nblk - 1);
  const int j = jb * 32;
  const int last = static_cast<int>(u.kv_len) - 1 - j;
  const uint32_t page = u.table[static_cast<uint32_t>(j) / a.page_tokens];
  const uint32_t slot0 = static_cast<uint32_t>(j) % a.page_tokens;
  const int8_t *vb = a.v + page * a.page_bytes + slot0 * a.row_bytes + u.kvh * HD;
  const int8_t *vsb = reinterpret_cast<const int8_t *>(a.vs) + page * a.scale_page_bytes + slot0 * a.scale_row_bytes;
  // the block's V rows into the wave's stage, then the score, scale and
  // block-maximum loads
  int8_t *st = vst[wave];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = 8 * e + (lane >> 3);
    lds_copy16(vb + min(r, last) * a.row_bytes + 16 * ((lane & 7) ^ vswz(r)), st + 1024 * e);
  }
  // lane = 32 h + key (scores), 32 h + block (maxima)
  const int c = lane & 31, h = lane >> 5;
  const int64_t wb = (static_cast<int64_t>(u.row) * a.heads + u.kvh * kGrp + h) * a.ldb;
  const float s = a.ws_s[(wb + jb) * 32 + c];
  const float vscale = reinterpret_cast<const float *>(vsb + min(c, last) * a.scale_row_bytes)[u.kvh];
  const float own = a.ws_bmax[wb + jb];
  // maximum of the blocks before this one (any order: scores are never NaN
  // nor -0, so the walk's select max is associative)
  float m = kFloor;
  for (int i = c; i < jb; i += 128) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = a.ws_bmax[wb + min(i + 32 * e, jb - 1)];
    m = fmaxf(m, fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
  }
  if (threadIdx.x == 0) stage_exp2_table(tab);
  wait_vmcnt<0>();  // the copies have landed
  __syncthreads();
  if (blk >= u.nblk) return;
  const float nmm = fmaxf(max32(m), own);
  float p = 0.0f, pv = 0.0f;
  if (c <= last) {
    p = exp_f32_le0_tab(__fsub_rn(s, nmm), tab);
    pv = __fmul_rn(p, vscale);
  }
  const float psum = tree_sum32(p);
  const float pm = __fmul_rn(max32(pv), inv127());
  p8s[wave][h][p8_pos(c)] = static_cast<int8_t>(quant1(pv, pm));
  if (c == 0) {
    a.ws_psum[wb + jb] = psum;
    a.ws_nmm[wb + jb] = nmm;
  }
  // P8.V (k_attn_decode.hip pv_mfma): A row m carries head m % 2's P8, so
  // result register q of every lane holds head q % 2, dim 16 t + lane % 16;
  // each 16-lane group stores two of the eight dim tiles
  const int tr_key = 16 * (((lane & 15) >> 1) >> 2) + 4 * (lane >> 4) + (((lane & 15) >> 1) & 3);
  const int tr_base = tr_key * HD + 8 * (lane & 1);
  const int tr_sw = vswz(tr_key);
  const float pm0 = lane_bcast<0>(pm), pm1 = lane_bcast<32>(pm);
  const long av = *reinterpret_cast<const long *>(p8s[wave][lane & 1] + 8 * (lane >> 4));
  const v4i_d z = {0, 0, 0, 0};
  v4i_d acc[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const v2i_d bt = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
        reinterpret_cast<lds_v2i_ptr_d>(to_lds(st + tr_base + ((t ^ tr_sw) << 4))));
    long bv;
    __builtin_memcpy(&bv, &bt, sizeof(bv));
    acc[t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bv, z, 0, 0, 0);
  }
  const int g = lane >> 4;
  float *dst = a.ws_pv + ((static_cast<int64_t>(u.row) * a.heads + u.kvh * kGrp) * a.ldb + jb) * HD;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    int i0 = acc[4 * q][0], i1 = acc[4 * q][1];
#pragma unroll
    for (int e = 1; e < 4; ++e) {
      i0 = g == e ? acc[4 * q + e][0] : i0;
      i1 = g == e ? acc[4 * q + e][1] : i1;
    }
    const int d = 64 * q + lane;
    dst[d] = __fmul_rn(static_cast<float>(i0), pm0);
    dst[static_cast<int64_t>(a.ldb) * HD + d] = __fmul_rn(static_cast<float>(i1), pm1);
  }
}

// ---- several rows of one sequence (a short chunk) ---------------------------
// The rows' int8 Q and K/V pages are there already, so both launches before
// the chain work on (16-row tile, KV head, 4 blocks): PV = false the block
// maxima of every row, PV = true the scores once more (four MFMAs a block cost
// less than 2 KiB of scores through memory), then P, psum, P8 and P8.V.  Lane
// layout of k_attn_prefill.hip: S^T = K.Q^T, lane (lc, lg) holds keys 16 kt +
// 4 lg + i of row lc, whose P8 bytes are the B operand of V^T.P8^T.
// What bounds it: latency at one tile (37 rows x 1040 keys: maxima 5.2, pv 12.2,
// chain 7.0 us, the walk 24.6), the pv blocks (8 KiB a tile and head) through
// memory from a few tiles on.  One query head per wave was faster for up to 8
// rows (4000 keys 1574 against 1596 us a chunk) and slower from 37 on (2202
// against 2112).
constexpr int kTile = 16;

template <bool PV>
__global__ void __launch_bounds__(kWaves * 64) split_chunk_kernel(SplitArgs a) {
  __shared__ uint64_t tab[32];
  __shared__ __align__(16) int8_t vst[PV ? kWaves : 1][32 * HD];
  __shared__ __align__(16) float scs[kWaves][64];
  // ids with equal residues mod 8 (one XCD) take the KV heads and tiles of a run
  const int ntiles = (a.rows + kTile - 1) / kTile;
  const int id = static_cast<int>(blockIdx.x);
  const int t = id >> 3;
  const int kvh = t % a.kv_heads;
  const int qi = t / a.kv_heads % ntiles * kTile;
  const int b0 = (t / (a.kv_heads * ntiles) * 8 + (id & 7)) * kWaves;
  const int nr = min(kTile, a.rows - qi);
  const int kv_len = static_cast<int>(a.kv_len);
  const int pos0 = kv_len - a.rows + qi;
  const int nblk = (pos0 + nr + 31) / 32;
  if (b0 >= nblk) return;
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int lc = lane & 15, lg = lane >> 4;
  const int blk = b0 + wave;
  const int jb = min(blk, nblk - 1);
  const int j = jb * 32;
  const int row = qi + min(lc, nr - 1);  // (lanes past the tile's rows repeat the last)
  const uint32_t page = a.table[static_cast<uint32_t>(j) / a.page_tokens];
  const uint32_t slot0 = static_cast<uint32_t>(j) % a.page_tokens;
  const int64_t koff = page * a.page_bytes + slot0 * a.row_bytes + kvh * HD;
  if constexpr (PV) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 8 * e + (lane >> 3);
      lds_copy16(a.v + koff + r * a.row_bytes + 16 * ((lane & 7) ^ vswz(r)), vst[wave] + 1024 * e);
    }
  }
  v4i_d kop[2][2], qop[kGrp][2];
  float qsv[kGrp];
#pragma unroll
  for (int kt = 0; kt < 2; ++kt)
#pragma unroll
    for (int k = 0; k < 2; ++k)
      kop[kt][k] = *reinterpret_cast<const v4i_d *>(a.k + koff + (16 * kt + lc) * a.row_bytes + 16 * lg + 64 * k);
#pragma unroll
  for (int h = 0; h < kGrp; ++h) {
    const int qh = kvh * kGrp + h;
#pragma unroll
    for (int k = 0; k < 2; ++k)
      qop[h][k] = *reinterpret_cast<const v4i_d *>(a.q8 + row * a.ldq8 + qh * HD + 16 * lg + 64 * k);
    qsv[h] = a.qs[row * a.ldqs + qh];
  }
  // lanes 0-31 the keys' ks, 32-63 their vs (0 past kv_len)
  const int8_t *sb = reinterpret_cast<const int8_t *>(lane < 32 ? a.ks : a.vs) + page * a.scale_page_bytes +
                     slot0 * a.scale_row_bytes;
  const float scv = reinterpret_cast<const float *>(sb + (lane & 31) * a.scale_row_bytes)[kvh];
  // row lc's maximum over the blocks before b0 (lane lg every fourth run), and
  // the run's own blocks
  float mrun[kGrp];
  float4 grp[kGrp];
  if constexpr (PV) {
#pragma unroll
    for (int h = 0; h < kGrp; ++h) {
      const float *bm = a.ws_bmax + (static_cast<int64_t>(row) * a.heads + kvh * kGrp + h) * a.ldb;
      grp[h] = *reinterpret_cast<const float4 *>(bm + b0);
      float m = kFloor;
      for (int i = 4 * lg; i < b0; i += 16) {
        const float4 v = *reinterpret_cast<const float4 *>(bm + i);
        m = fmaxf(m, fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)));
      }
      mrun[h] = m;
    }
    if (threadIdx.x == 0) stage_exp2_table(tab);
  }
  float *sc = scs[wave];
  sc[lane] = j + (lane & 31) < kv_len ? scv : 0.0f;
  if constexpr (PV) {
    wait_vmcnt<0>();  // the V copies have landed
    __syncthreads();
  }
  if (blk >= nblk) return;
  float ksr[2][4], vsr[2][4];
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    const float4 k4 = *reinterpret_cast<const float4 *>(sc + 16 * kt + 4 * lg);
    const float4 v4 = *reinterpret_cast<const float4 *>(sc + 32 + 16 * kt + 4 * lg);
    ksr[kt][0] = k4.x, ksr[kt][1] = k4.y, ksr[kt][2] = k4.z, ksr[kt][3] = k4.w;
    vsr[kt][0] = v4.x, vsr[kt][1] = v4.y, vsr[kt][2] = v4.z, vsr[kt][3] = v4.w;
  }
  const v4i_d z = {0, 0, 0, 0};
  auto fold_max = [](float v) {  // over the four lanes of a row
    LanePair p = lane_pair16(__float_as_uint(v));
    v = fmaxf(__uint_as_float(p.a), __uint_as_float(p.b));
    p = lane_pair32(__float_as_uint(v));
    return fmaxf(__uint_as_float(p.a), __uint_as_float(p.b));
  };
#pragma unroll
  for (int h = 0; h < kGrp; ++h) {
    float s[2][4], bmax = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      v4i_d acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(kop[kt][0], qop[h][0], z, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(kop[kt][1], qop[h][1], acc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = __fmul_rn(static_cast<float>(acc[i]), ksr[kt][i]);
        x = __fmul_rn(x, qsv[h]);
        x = __fmul_rn(x, a.qk_scale);
        if (j + 16 * kt + 4 * lg + i > pos0 + lc) x = -INFINITY;
        s[kt][i] = x;
        bmax = fmaxf(bmax, x);
      }
    }
    bmax = fold_max(bmax);
    const int64_t wb = (static_cast<int64_t>(row) * a.heads + kvh * kGrp + h) * a.ldb + blk;
    if constexpr (!PV) {
      if (lg == 0 && lc < nr) a.ws_bmax[wb] = bmax;
    } else {
      float nmm = fmaxf(fold_max(mrun[h]), bmax);
      if (wave > 0) nmm = fmaxf(nmm, grp[h].x);
      if (wave > 1) nmm = fmaxf(nmm, grp[h].y);
      if (wave > 2) nmm = fmaxf(nmm, grp[h].z);
      float p[2][4], ts[2], pmx = 0.0f;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) p[kt][i] = exp_f32_le0_fast(__fsub_rn(s[kt][i], nmm), tab);
        // the pairwise tree over the 32 keys: key bits 0-1 in registers, bits
        // 2 and 3 over lg, bit 4 = kt
        float u = __fadd_rn(__fadd_rn(p[kt][0], p[kt][1]), __fadd_rn(p[kt][2], p[kt][3]));
        LanePair q = lane_pair16(__float_as_uint(u));
        u = __fadd_rn(__uint_as_float(q.a), __uint_as_float(q.b));
        q = lane_pair32(__float_as_uint(u));
        ts[kt] = __fadd_rn(__uint_as_float(q.a), __uint_as_float(q.b));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[kt][i] = __fmul_rn(p[kt][i], vsr[kt][i]);
          pmx = fmaxf(pmx, p[kt][i]);
        }
      }
      const float pm = __fmul_rn(fold_max(pmx), inv127());
      const double y = rcp64(pm);
      // (as k_attn_prefill.hip quantises: without clamps while every row's pm is
      // normal, so that a negative vs, which no quantisation gives, comes out
      // the same on both routes)
      uint32_t q8[2][4], w8[2];
      if (__builtin_amdgcn_ballot_w64(!(pm >= 1.17549435e-38f)) == 0) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            q8[kt][i] = static_cast<uint32_t>(
                static_cast<int>(rintf(__double2float_rn(__dmul_rn(static_cast<double>(p[kt][i]), y)))));
      } else {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) q8[kt][i] = static_cast<uint32_t>(quant_rcp_pos(p[kt][i], y));
      }
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        w8[kt] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(q8[kt][3], q8[kt][2], 0x0c0c0400u),
                                       __builtin_amdgcn_perm(q8[kt][1], q8[kt][0], 0x0c0c0400u), 0x05040100u);
      if (lg == 0 && lc < nr) {
        a.ws_psum[wb] = __fadd_rn(ts[0], ts[1]);
        a.ws_nmm[wb] = nmm;
      }
      const long bp = static_cast<long>((static_cast<uint64_t>(w8[1]) << 32) | w8[0]);
      const int jj = (lane & 15) >> 1;
      const int key = 16 * (jj >> 2) + 4 * lg + (jj & 3);
      const int8_t *vq = vst[wave] + key * HD + 8 * (lane & 1);
      float *dst = a.ws_pv + wb * HD + 4 * lg;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        const v2i_d vt =
            __builtin_amdgcn_ds_read_tr8_b64_v2i32(reinterpret_cast<lds_v2i_ptr_d>(to_lds(vq + ((dt ^ vswz(key)) << 4))));
        long va;
        __builtin_memcpy(&va, &vt, sizeof(va));
        const v4i_d c = __builtin_amdgcn_mfma_i32_16x16x32_i8(va, bp, z, 0, 0, 0);
        if (lc < nr)
          *reinterpret_cast<float4 *>(dst + 16 * dt) =
              make_float4(__fmul_rn(static_cast<float>(c[0]), pm), __fmul_rn(static_cast<float>(c[1]), pm),
                          __fmul_rn(static_cast<float>(c[2]), pm), __fmul_rn(static_cast<float>(c[3]), pm));
      }
    }
  }
}

constexpr int kChainWaves = 8;
constexpr int kStage = 16;        // blocks per LDS stage (one instruction per wave)
constexpr int kStages = 8;        // stages in flight
constexpr int kChainBlocks = kStage * kStages;

__global__ void __launch_bounds__(kChainWaves * 64) split_chain_kernel(SplitArgs a) {
  __shared__ uint64_t tab[32];
  __shared__ __align__(16) float pvs[kChainBlocks][HD];
  __shared__ float amax[2];
  const int row = static_cast<int>(blockIdx.x) / a.heads;
  const int qh = static_cast<int>(blockIdx.x) % a.heads;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = wave_id();
  const uint32_t kv_len = a.row_pos ? static_cast<uint32_t>(a.row_pos[row]) + 1 : a.kv_len - (a.rows - 1 - row);
  const int nblk = static_cast<int>((kv_len + 31) / 32);
  const int64_t wb = (static_cast<int64_t>(row) * a.heads + qh) * a.ldb;
  if (tid == 0) stage_exp2_table(tab);
  float res = 0.0f, den = 0.0f;
  for (int b0 = 0; b0 < nblk; b0 += kChainBlocks) {
    const int nb = min(kChainBlocks, nblk - b0);
    // waves 0, 1: lane l's blocks b0 + 64 q + l: maximum, the one before, psum
    float nm[2], pm[2], ps[2], corr[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int jl = b0 + min(64 * q + lane, nb - 1);
      nm[q] = a.ws_nmm[wb + jl];
      pm[q] = a.ws_nmm[wb + max(jl - 1, 0)];
      if (jl == 0) pm[q] = kFloor;
      ps[q] = a.ws_psum[wb + jl];
    }
    // pv rows, 2 blocks per instruction (past the chunk: its last block);
    // stages past the chunk are not copied
#pragma unroll
    for (int e = 0; e < kStages; ++e) {
      if (kStage * e < nb) {
        const int j = kStage * e + 2 * wave;
        const int blk = b0 + min(j + (lane >> 5), nb - 1);
        lds_copy16(a.ws_pv + (wb + blk) * HD + 4 * (lane & 31), &pvs[j][0]);
      }
    }
    const bool full = nb > kStage * (kStages - 1);  // every stage was copied
    // stage e is complete once every wave's own copy of it has landed (one
    // wait for all of a partial chunk)
    static_for<kStages>([&](auto E) {
      constexpr int e = decltype(E)::value;
      if (kStage * e >= nb) return;
      if (full) {
        wait_vmcnt<kStages - 1 - e>();
        lds_barrier();
      } else if (e == 0) {
        wait_vmcnt<0>();
        lds_barrier();
      }
      if (wave < 2) {
        constexpr int q = kStage * e / 64, l0 = kStage * e % 64;
        if (l0 == 0) corr[q] = exp_f32_le0_tab(__fsub_rn(pm[q], nm[q]), tab);
        float pw[kStage];
#pragma unroll
        for (int i = 0; i < kStage; ++i) pw[i] = pvs[kStage * e + i][tid];
#pragma unroll
        for (int i = 0; i < kStage; ++i) {
          if (kStage * e + i < nb) {
            const float cr = lane_read(corr[q], l0 + i);
            den = __fadd_rn(__fmul_rn(den, cr), lane_read(ps[q], l0 + i));
            res = __fadd_rn(__fmul_rn(res, cr), pw[i]);
          }
        }
      }
    });
    if (b0 + kChainBlocks < nblk) {
      wait_vmcnt<0>();
      lds_barrier();  // the stages are free again
    }
  }
  // a chunk's rows walk to the end of their 32-row block's last row
  // (ref_qwen3.py:281-288): fully masked blocks add +0 to res (-0 becomes +0)
  if (!a.row_pos && static_cast<int>((kv_len + (min(row | 31, a.rows - 1) - row) + 31) / 32) > nblk)
    res = __fadd_rn(res, 0.0f);
  // ---- epilogue: out = res * (1/den); per-head int8 quant (522-546) ----
  float out = 0.0f;
  if (wave < 2) {
    out = __fmul_rn(res, __fdiv_rn(1.0f, den));
    float mx = max64(fabsf(out));
    // a chunk's row without a number (infinite or NaN scores) gets scale 0 as
    // from k_attn_prefill.hip, a decoding row NaN as from k_attn_decode.hip
    if (!a.row_pos && a.rows > 1) mx = fmaxf(mx, 0.0f);
    if (lane == 0) amax[wave] = mx;
  }
  wait_vmcnt<0>();
  lds_barrier();
  if (wave < 2) {
    const float scale = __fmul_rn(fmaxf(amax[0], amax[1]), inv127());
    a.o8[static_cast<int64_t>(row) * a.ldo + qh * HD + tid] = static_cast<int8_t>(quant1(out, scale));
    if (tid == 0) a.os[static_cast<int64_t>(row) * a.ldos + qh] = scale;
  }
}

}  // namespace

bool attn_split_supported(const SplitArgs &a) {
  auto al16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (a.rows < 1 || a.kv_heads < 1 || a.heads != kGrp * a.kv_heads || a.max_blocks < 1 || a.ldb < a.max_blocks)
    return false;
  if (a.page_tokens % 32 || a.row_bytes % 16 || a.page_bytes % 16 || a.scale_row_bytes % 4 || !al16(a.k) || !al16(a.v))
    return false;
  if (!a.ws_s || !a.ws_bmax || !a.ws_nmm || !a.ws_psum || !a.ws_pv || !al16(a.ws_pv)) return false;
  return true;
}

// A batch takes the split when the single launch's serial walk of its longest
// row (~0.53 us per block past the first chunk) costs more than the split's
// work over all rows (~0.016 us per row and block) and its extra launches.
// Measured on the 28-layer decode step, us (single launch / split):
// 1 row x 384 keys 1127 / 1099, 1 x 2048 1942 / 1168, 5 x 700 1469 / 1306,
// 16 x 384 1339 / 1371, 16 x 2048 2210 / 1745, 24 x 700 1579 / 1560, 32 x
// 1024 1784 / 1789, 32 x 2048 2349 / 2217, 48 x 2048 2665 / 2795, 64 x 2048
// 2854 / 3308.
bool attn_split_batch(int64_t max_blocks, int64_t sum_blocks) {
  return max_blocks >= 12 && 36 * max_blocks > sum_blocks + 250;
}

hipError_t launch_attn_split(const SplitArgs &a, hipStream_t s) {
  if (!attn_split_supported(a)) return hipErrorInvalidValue;
  const int64_t units = static_cast<int64_t>(a.rows) * ((a.max_blocks + kWaves - 1) / kWaves);
  const int64_t grid = (units + 7) / 8 * 8 * a.kv_heads;
  if (grid >= (int64_t{1} << 31)) return hipErrorInvalidValue;
  Q3_LAUNCH(split_score_kernel, dim3(static_cast<unsigned>(grid)), dim3(kWaves * 64), 0, s, a);
  Q3_LAUNCH(split_pv_kernel, dim3(static_cast<unsigned>(grid)), dim3(kWaves * 64), 0, s, a);
  Q3_LAUNCH(split_chain_kernel, dim3(static_cast<unsigned>(a.rows * a.heads)), dim3(kChainWaves * 64), 0, s, a);
  return hipGetLastError();
}

bool attn_split_chunk_supported(const SplitArgs &a) {
  if (!attn_split_supported(a) || a.row_pos || a.ldb % 4) return false;
  if (a.kv_len < static_cast<uint32_t>(a.rows) || static_cast<int64_t>(a.max_blocks) * 32 < a.kv_len) return false;
  auto al16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  return al16(a.q8) && a.ldq8 % 16 == 0 && al16(a.ws_bmax);
}

// A chunk takes the split when the prefill kernel's walk (one workgroup per
// 16-row tile and head, ~0.5 us per block) is long beside what every tile adds
// to the split, its pv blocks through memory (~3 us a tile at 64 blocks).
// 28-layer chunks, us (walk / split): 2 rows x 640 keys 1131 / 1148, 800 1235
// / 1155, 2048 1804 / 1202, 4000 2790 / 1297; 16 x 800 1529 / 1491, 4000 3128
// / 1716; 17 x 800 1558 / 1565, 1040 1685 / 1592; 37 x 1040 1722 / 1743, 1500
// 1912 / 1849, 4000 3128 / 2112; 64 x 1040 1773 / 1818, 1500 1962 / 1939, 4000
// 3172 / 2407; 96 x 2048 2402 / 2404, 128 x 2048 2393 / 2620.
bool attn_split_chunk(int64_t rows, int64_t nblocks) {
  return rows <= 64 && nblocks >= 17 + 8 * ((rows + kTile - 1) / kTile);
}

hipError_t launch_attn_split_chunk(const SplitArgs &a, hipStream_t s) {
  if (!attn_split_chunk_supported(a)) return hipErrorInvalidValue;
  const int64_t runs = (a.max_blocks + kWaves - 1) / kWaves, tiles = (a.rows + kTile - 1) / kTile;
  const int64_t grid = (runs + 7) / 8 * 8 * a.kv_heads * tiles;
  if (grid >= (int64_t{1} << 31)) return hipErrorInvalidValue;
  Q3_LAUNCH(split_chunk_kernel<false>, dim3(static_cast<unsigned>(grid)), dim3(kWaves * 64), 0, s, a);
  Q3_LAUNCH(split_chunk_kernel<true>, dim3(static_cast<unsigned>(grid)), dim3(kWaves * 64), 0, s, a);
  Q3_LAUNCH(split_chain_kernel, dim3(static_cast<unsigned>(a.rows * a.heads)), dim3(kChainWaves * 64), 0, s, a);
  return hipGetLastError();
}

}  // namespace q3
