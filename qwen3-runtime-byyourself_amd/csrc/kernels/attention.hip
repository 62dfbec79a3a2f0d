// Causal grouped-query attention for gfx950 (src/ops/gqa_attention.cu:20-155
// of the reference: query [B, S, Hq * D], key/value cache views
// [B, cached, Hkv, D] with strides, query (b, s) attends to keys
// 0 .. start + s, query head h reads KV head h / (Hq / Hkv)).
//
// Matrix-core path (head_dim 128, unit dim stride, 16-byte rows): a block of
// four waves owns one (batch, KV head) and 128 of its (position, head)
// columns, so every K/V tile it stages in LDS serves 128 query rows.  (A
// prefill too short to fill the GPU that way takes blocks of eight waves whose
// two or four groups divide the keys of the same columns and merge in LDS;
// attention of at most 32 columns, decode above all, a kernel of its own whose
// waves share nothing: dispatch.hpp.)  A wave's
// 32 "columns" are consecutive (position, head) pairs in position-major
// order: 32 / G whole positions when G divides 32; any G up to 32 works (for
// Qwen3-14B's 5 a position's heads may straddle two waves).  Per 32 keys:
//   S^T = K Q^T   with v_mfma_f32_32x32x16_bf16: A = K rows from LDS,
//                 B = the wave's Q fragments (registers for the whole loop);
//   online softmax per column: a lane holds one column, so the key max and
//                 sum need only its own registers and the lane 32 apart
//                 (v_permlane32_swap);
//   O^T += V^T P^T: A = V^T read from the row-major V tile with the LDS
//                 transpose read (ds_read_b64_tr_b16), B = P^T straight from
//                 the S^T registers.  P is split into a bf16 high part and a
//                 bf16 remainder (two MFMAs), so the weights keep about 16
//                 significant bits: the reference accumulates p * v in fp32,
//                 and a single bf16 rounding of p would cost up to half an
//                 output ulp.
// Scores are scaled by scale * log2(e) and exponentiated with v_exp_f32.
// Keys go in tiles of 64 (two S^T halves of 32).  A tile's K and V rows go
// from HBM straight into LDS (buffer_load_dwordx4 ... lds, no registers) while
// the previous tile is computed, into the other of two buffers; one barrier
// per tile.  The P V product of a tile is issued in the next tile's step,
// beside that tile's softmax.  One wave's independent MFMA and VALU work can
// overlap on gfx950, but interleaving them within the wave measured slower
// here than leaving the overlap to the other block's wave on the same SIMD
// (two waves per SIMD at this register count).  Tile rows are 256 bytes with
// the 16-byte chunks XOR-swizzled by row so that the K fragment reads
// (ds_read_b128) and the V transpose reads hit distinct LDS banks.
//
// Generic path (any head_dim <= 256, any strides): one wave per query row,
// keys in order, lanes over the head dimension -- the reference's own
// structure with wave reductions.
#include <type_traits>

#include "dispatch.hpp"
#include "q3k_common.hpp"

namespace q3k
{
    namespace
    {
        typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
        typedef float f32x16_t __attribute__((ext_vector_type(16)));

        typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) bf16x4_t lds_bf16x4_t;
        typedef __attribute__((address_space(3))) void lds_void_t;

        constexpr int kAttD = kAttHeadDim;
        constexpr int kRowBytes = kAttD * 2;                  // one K or V row in LDS
        constexpr int kRowsPerLoad = kWave * 16 / kRowBytes;  // rows one wave-wide 16-byte load fills
        constexpr int kAhead = 2;                             // LDS fragment reads in flight ahead of use
        constexpr float kLazyMax = 8.0f;                      // log2 headroom before the softmax reference moves
        constexpr float kLog2e = 1.4426950408889634f;

        struct AttnArgs
        {
            const uint16_t *q;
            const uint16_t *k;
            const uint16_t *v;
            uint16_t *out;
            int64_t S;
            int64_t start;
            int64_t ks0, ks1, ks2, ks3;
            int64_t vs0, vs1, vs2, vs3;
            int32_t Hq;
            int32_t Hkv;
            int32_t D;
            int32_t qblocks;
            float scale;
            // split-K: the key range is cut into at most `splits` slices of
            // split_keys keys (a multiple of the tile); a query block takes the
            // slices its causal range reaches.  With more than one, slice results
            // (unnormalised O^T, reference max and sum) go to part_o [splits,
            // rows, D] and part_ml [splits, rows, 2] and attn_combine_kernel
            // merges them
            int32_t splits;
            int32_t split_keys;
            float *part_o;
            float *part_ml;
            int64_t rows;
        };

        __device__ __forceinline__ bf16x8_t as_bf8(const Vec8 &v) { return __builtin_bit_cast(bf16x8_t, v); }

        // LDS chunk (16 bytes) holding chunk c of K row r / V row r of a tile.
        // K: lanes 0..31 of a fragment read read rows r..r+31 at one chunk;
        // any 16 consecutive rows put it in 16 different chunk positions.
        // V: a transpose read takes 4 rows x 32 bytes per 16 lanes; rows
        // 4 apart share a bank set.
        __device__ __forceinline__ int k_slot(int r, int c) { return c ^ (r & 15); }
        __device__ __forceinline__ int v_slot(int r, int c) { return c ^ (4 * (r & 3)); }

        // Buffer resource over [base, base + 2 GiB): raw (stride 0), so the
        // offsets the loads give are byte offsets from base.
        __device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const void *base)
        {
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, 0x7fffffff, 0x00020000);
        }

        // 16 bytes per lane from rsrc + voffset into LDS at lds_wave + 16 * lane
        // (buffer_load_dwordx4 ... lds: no registers, the wave's LDS base in M0)
        __device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, int32_t voffset, unsigned char *lds_wave)
        {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t *)lds_wave, 16, voffset, 0, 0, 0);
        }

        // max / sum of x over lanes l and l ^ 32, in every lane (one VALU swap,
        // no LDS): after the swap one operand is x and the other its partner
        __device__ __forceinline__ float pair_max(float x)
        {
            const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
            return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
        }
        __device__ __forceinline__ float pair_sum(float x)
        {
            const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
            return __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }

        // Waits until at most N of the wave's vector loads are in flight and its
        // LDS reads are done (s_waitcnt vmcnt(N) lgkmcnt(0); 63: the LDS reads only).
        template <int N>
        __device__ __forceinline__ void wait_loads()
        {
            static_assert(N >= 0 && N < 64, "vmcnt");
            __asm__ volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
            __asm__ volatile("" ::: "memory");
        }

        // ---- tile operations shared by the kernels ------------------------------

        // Loading a key tile's K (or V) rows into LDS by CW waves: wave cw fills
        // rows (KEYS / CW) cw .. of a buffer, kRowsPerLoad rows per load; lane j
        // lands in slot j % 16 of row j / 16 and so fetches the chunk that slot
        // holds.  A tile's loads address from a buffer resource based at its first
        // key, so the per-lane byte offsets (tile_offsets) stay fixed: 32-bit,
        // checked by the launcher.  Rows past n_keys repeat the last key (finite
        // data, later masked or weighted by zero).
        template <int CW, int KEYS>
        struct Staging
        {
            static constexpr int kRows = KEYS / CW;             // rows of a tile per wave
            static constexpr int kLoads = kRows / kRowsPerLoad; // loads per wave per K (or V) tile
        };

        template <int CW, int KEYS, typename Slot>
        __device__ __forceinline__ void tile_offsets(int cw, int lane, int32_t byte_stride, Slot slot,
                                                     int32_t (&voff)[Staging<CW, KEYS>::kLoads])
        {
            const int st_row = Staging<CW, KEYS>::kRows * cw + lane / 16;
#pragma unroll
            for (int x = 0; x < Staging<CW, KEYS>::kLoads; ++x)
            {
                const int r = st_row + kRowsPerLoad * x;
                voff[x] = r * byte_stride + 16 * slot(r, lane % 16);
            }
        }

        template <int CW, int KEYS, typename Slot>
        __device__ __forceinline__ void load_tile_rows(int tile, unsigned char *buf, const uint16_t *base,
                                                       int64_t row_stride, int32_t byte_stride, int32_t n_keys, int cw,
                                                       int lane, const int32_t (&voff)[Staging<CW, KEYS>::kLoads],
                                                       Slot slot)
        {
            constexpr int kRows = Staging<CW, KEYS>::kRows;
            const int32_t key0 = tile * KEYS;
            const __amdgpu_buffer_rsrc_t rs = tile_rsrc(base + static_cast<int64_t>(key0) * row_stride);
            unsigned char *dst = buf + kRows * cw * kRowBytes;
            if (key0 + KEYS <= n_keys)
            {
#pragma unroll
                for (int x = 0; x < Staging<CW, KEYS>::kLoads; ++x)
                    dma16(rs, voff[x], dst + kRowsPerLoad * x * kRowBytes);
            }
            else
            {
                const int last = n_keys - 1 - key0;
                const int st_row = kRows * cw + lane / 16;
#pragma unroll
                for (int x = 0; x < Staging<CW, KEYS>::kLoads; ++x)
                {
                    const int r = st_row + kRowsPerLoad * x;
                    const int rr = r < last ? r : last;
                    dma16(rs, rr * byte_stride + 16 * slot(r, lane % 16), dst + kRowsPerLoad * x * kRowBytes);
                }
            }
        }

        // Q fragments of the lane's column.  A padding column (s_col >= S) reads
        // the last position's row instead: its scores are always masked (a wave
        // holding one is a partial wave), so only finiteness matters.
        __device__ __forceinline__ void load_q(const AttnArgs &a, int64_t b, int32_t s_col, int h_col, bool col_ok,
                                               int lg, bf16x8_t (&qf)[kAttD / 16])
        {
            const int64_t s_row = col_ok ? s_col : a.S - 1;
            const Vec8 *qrow = reinterpret_cast<const Vec8 *>(a.q + ((b * a.S + s_row) * a.Hq + h_col) * kAttD);
#pragma unroll
            for (int c = 0; c < kAttD / 16; ++c)
                qf[c] = as_bf8(qrow[2 * c + lg]);
        }

        // Per-lane LDS byte offsets of the V transpose reads: the lanes of each
        // 16 give rows 4 lg + j / 4 (+ 8 per 8-key step) and 4 dims
        // 32 dt + 16 ((lane / 16) % 2) + 4 (j % 4) .. + 3, and each lane gets 4
        // consecutive keys of one dim (dim 32 dt + lane % 32).
        __device__ __forceinline__ void v_offsets(int lane, int (&v_off)[kAttD / 32])
        {
            const int tj = lane % 16, lg = lane / 32;
            const int v_row = 4 * lg + tj / 4;
#pragma unroll
            for (int dt = 0; dt < kAttD / 32; ++dt)
                v_off[dt] = v_row * kRowBytes + 16 * v_slot(v_row, 4 * dt + 2 * ((lane / 16) % 2) + (tj % 4) / 2) +
                            8 * (tj % 2);
        }

        // The V^T fragment of P V step i (key chunk i / 4, dims 32 (i % 4) .. + 31):
        // keys 16 (i / 4) + 8 t + 4 lg + 0..3 in elements 4 t .. 4 t + 3, the keys
        // of the P^T elements this lane holds.
        __device__ __forceinline__ bf16x8_t read_v(const unsigned char *v_lds, const int (&v_off)[kAttD / 32], int i)
        {
            const unsigned char *vp = v_lds + v_off[i % 4] + 16 * (i / 4) * kRowBytes;
            const bf16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_t *)(vp));
            const bf16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_t *)(vp + 8 * kRowBytes));
            return __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
        }

        // S^T = K Q^T for the 32 HH keys of a tile (sacc[hh]: keys 32 hh .. + 31).
        // The K fragment reads run kAhead steps ahead of the MFMAs that use them.
        // When its own reads have run out it calls next(x), x < kAhead, for the
        // reads of the product that follows.
        template <int HH, typename Next>
        __device__ __forceinline__ void qk_tile(const unsigned char *k_lds, const bf16x8_t (&qf)[kAttD / 16], int li,
                                                int lg, f32x16_t (&sacc)[HH], Next next)
        {
            auto read_k = [&](int c, int hh) __attribute__((always_inline)) {
                return *reinterpret_cast<const Vec8 *>(k_lds + (32 * hh + li) * kRowBytes +
                                                       16 * k_slot(li, 2 * c + lg));
            };
#pragma unroll
            for (int hh = 0; hh < HH; ++hh)
                sacc[hh] = f32x16_t{};
            Vec8 kq[kAhead + 1][HH];
#pragma unroll
            for (int c = 0; c < kAhead; ++c)
#pragma unroll
                for (int hh = 0; hh < HH; ++hh)
                    kq[c][hh] = read_k(c, hh);
#pragma unroll
            for (int c = 0; c < kAttD / 16; ++c)
            {
                if (c + kAhead < kAttD / 16)
#pragma unroll
                    for (int hh = 0; hh < HH; ++hh)
                        kq[(c + kAhead) % (kAhead + 1)][hh] = read_k(c + kAhead, hh);
                if (c + kAhead >= kAttD / 16)
                    next(c + kAhead - kAttD / 16);
                __builtin_amdgcn_sched_barrier(0); // keep the reads ahead of these MFMAs
#pragma unroll
                for (int hh = 0; hh < HH; ++hh)
                    sacc[hh] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(kq[c % (kAhead + 1)][hh]), qf[c], sacc[hh],
                                                                       0, 0, 0);
            }
        }

        // Scores of keys past the column's causal limit and of padding columns
        // become -inf (before the max).
        template <int HH>
        __device__ __forceinline__ void mask_tile(f32x16_t (&sacc)[HH], int32_t key0, int lg, int32_t last_key,
                                                  bool col_ok)
        {
#pragma unroll
            for (int hh = 0; hh < HH; ++hh)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                {
                    const int32_t kk = key0 + 32 * hh + 8 * (r / 4) + 4 * lg + (r % 4);
                    if (kk > last_key || !col_ok)
                        sacc[hh][r] = -__builtin_huge_valf();
                }
        }

        // Online softmax of one tile for the lane's column: the weights, split
        // into bf16 high parts and remainders, go to phi / plo, and m, l are
        // updated.  The weights are taken relative to a reference m that moves
        // only when a tile's max exceeds it by more than kLazyMax (log2 units):
        // they stay below 2^kLazyMax, and the rescale of the output is left for
        // the rare tiles that move it.  Returns that rescale factor (1 when m did
        // not move).  An all-masked column keeps m = -inf and weight 0.  The max
        // of the raw scores times the (positive) scale is the max of the scaled
        // ones.
        template <int HH>
        __device__ __forceinline__ float softmax_tile(const f32x16_t (&sacc)[HH], float scale2, float &m, float &l,
                                                      bf16x8_t (&phi)[HH][2], bf16x8_t (&plo)[HH][2])
        {
            float mloc = sacc[0][0];
#pragma unroll
            for (int hh = 0; hh < HH; ++hh)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    mloc = fmaxf(mloc, sacc[hh][r]);
            mloc = pair_max(mloc);
            const float m_tile = mloc * scale2;
            const bool move = m_tile > m + kLazyMax;
            const float m_new = move ? m_tile : m;
            const float m_use = m_new == -__builtin_huge_valf() ? 0.0f : m_new;
            const float alpha = move ? __builtin_amdgcn_exp2f(m - m_use) : 1.0f;
            float psum = 0.0f;
#pragma unroll
            for (int hh = 0; hh < HH; ++hh)
#pragma unroll
                for (int mm = 0; mm < 2; ++mm)
                {
                    Vec8 h8, l8;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                    {
                        const float x0 =
                            __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[hh][8 * mm + 2 * j], scale2, -m_use));
                        const float x1 =
                            __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[hh][8 * mm + 2 * j + 1], scale2, -m_use));
                        psum += x0;
                        psum += x1;
                        const uint32_t hp = pack_rne(x0, x1);
                        h8.d[j] = hp;
                        l8.d[j] = pack_rne(x0 - bf_lo(hp), x1 - bf_hi(hp));
                    }
                    phi[hh][mm] = as_bf8(h8);
                    plo[hh][mm] = as_bf8(l8);
                }
            psum = pair_sum(psum);
            l = l * alpha + psum;
            m = m_new;
            return alpha;
        }

        // o *= alpha; multiplying by alpha == 1 changes nothing, so the wave
        // skips it when no lane needs it
        __device__ __forceinline__ void rescale(f32x16_t (&o)[kAttD / 32], float alpha)
        {
            if (__any(alpha != 1.0f))
            {
#pragma unroll
                for (int dt = 0; dt < kAttD / 32; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        o[dt][r] *= alpha;
            }
        }

        // O^T += V^T P^T for one tile: step i covers the 16-key chunk i / 4
        // (hh = i / 8, mm = (i / 4) % 2) and dims 32 (i % 4) .. + 31.  The
        // transpose reads run kAhead steps ahead of the MFMAs that use them; the
        // first kAhead are in vq already.
        template <int HH>
        __device__ __forceinline__ void pv_tile(const unsigned char *v_lds, const int (&v_off)[kAttD / 32],
                                                const bf16x8_t (&phi)[HH][2], const bf16x8_t (&plo)[HH][2],
                                                f32x16_t (&o)[kAttD / 32], bf16x8_t (&vq)[kAhead + 1])
        {
#pragma unroll
            for (int i = 0; i < 8 * HH; ++i)
            {
                if (i + kAhead < 8 * HH)
                    vq[(i + kAhead) % (kAhead + 1)] = read_v(v_lds, v_off, i + kAhead);
                __builtin_amdgcn_sched_barrier(0); // keep the reads ahead of these MFMAs
                const int dt = i % 4, hh = i / 8, mm = (i / 4) % 2;
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vq[i % (kAhead + 1)], phi[hh][mm], o[dt], 0, 0, 0);
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vq[i % (kAhead + 1)], plo[hh][mm], o[dt], 0, 0, 0);
            }
        }

        // Dims 32 dt .. + 31 of the lane's column of the result: bf16 O / l, or
        // with split keys the slice's unnormalised O^T for the merge (and, once
        // per column, its reference max and sum: store_ml).
        __device__ __forceinline__ void store_dims(const AttnArgs &a, bool split, int sp, int64_t row, int dt, int lg,
                                                   const f32x16_t &o, float inv)
        {
            if (split)
            {
                float *po = a.part_o + (static_cast<int64_t>(sp) * a.rows + row) * kAttD;
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4)
                {
                    const float4 w = {o[4 * q4], o[4 * q4 + 1], o[4 * q4 + 2], o[4 * q4 + 3]};
                    *reinterpret_cast<float4 *>(po + dt * 32 + 8 * q4 + 4 * lg) = w;
                }
                return;
            }
            uint16_t *orow = a.out + row * kAttD;
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
            {
                uint2 w;
                w.x = pack_rne(o[4 * q4] * inv, o[4 * q4 + 1] * inv);
                w.y = pack_rne(o[4 * q4 + 2] * inv, o[4 * q4 + 3] * inv);
                *reinterpret_cast<uint2 *>(orow + dt * 32 + 8 * q4 + 4 * lg) = w;
            }
        }
        __device__ __forceinline__ void store_ml(const AttnArgs &a, int sp, int64_t row, float m, float l)
        {
            reinterpret_cast<float2 *>(a.part_ml)[static_cast<int64_t>(sp) * a.rows + row] = make_float2(m, l);
        }

        // The whole column of one wave.
        __device__ __forceinline__ void store_column(const AttnArgs &a, bool split, int sp, int64_t row, bool col_ok,
                                                     int lg, const f32x16_t (&o)[kAttD / 32], float m, float l)
        {
            if (!col_ok)
                return;
            const float inv = 1.0f / l;
#pragma unroll
            for (int dt = 0; dt < kAttD / 32; ++dt)
                store_dims(a, split, sp, row, dt, lg, o[dt], inv);
            if (split && lg == 0)
                store_ml(a, sp, row, m, l);
        }

        // The KW groups' partial results of a column meet in LDS, in the tile
        // buffers: dims 32 dt .. + 31 of all waves in buffer dt (4 KiB a wave, 16
        // bytes a lane, so lanes hit distinct banks).  Group kw then merges and
        // stores 4 / KW of the four parts.
        template <int CW, int KW>
        __device__ __forceinline__ void merge_groups(unsigned char *b0, unsigned char *b1, unsigned char *b2,
                                                     unsigned char *b3, const AttnArgs &a, bool split, int sp, int64_t row,
                                                     bool col_ok, int cw, int kw, int li, int lg,
                                                     const f32x16_t (&o)[kAttD / 32], float m, float l)
        {
            static_assert(kAttD / 32 == 4 && 4 % KW == 0, "parts");
            constexpr int kParts = 4 / KW;
            const int lane = 32 * lg + li, wave = kw * CW + cw;
            __shared__ float2 ml[KW][32 * CW];
            unsigned char *const bufs[4] = {b0, b1, b2, b3};
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
            {
                float4 *dst = reinterpret_cast<float4 *>(bufs[dt]) + wave * 4 * kWave;
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4)
                    dst[q4 * kWave + lane] = {o[dt][4 * q4], o[dt][4 * q4 + 1], o[dt][4 * q4 + 2], o[dt][4 * q4 + 3]};
            }
            if (lg == 0)
                ml[kw][32 * cw + li] = make_float2(m, l);
            __syncthreads();
            float w[KW];
            float mx = -__builtin_huge_valf();
#pragma unroll
            for (int x = 0; x < KW; ++x)
                mx = fmaxf(mx, ml[x][32 * cw + li].x);
            const float m_use = mx == -__builtin_huge_valf() ? 0.0f : mx;
            float lsum = 0.0f;
#pragma unroll
            for (int x = 0; x < KW; ++x)
            {
                const float2 e = ml[x][32 * cw + li];
                w[x] = __builtin_amdgcn_exp2f(e.x - m_use);
                lsum += w[x] * e.y;
            }
            const float inv = 1.0f / lsum;
#pragma unroll
            for (int y = 0; y < kParts; ++y)
            {
                const int dt = kw * kParts + y;
                const unsigned char *buf = dt == 0 ? b0 : dt == 1 ? b1 : dt == 2 ? b2 : b3;
                f32x16_t r = f32x16_t{};
#pragma unroll
                for (int x = 0; x < KW; ++x)
                {
                    const float4 *src = reinterpret_cast<const float4 *>(buf) + (x * CW + cw) * 4 * kWave;
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4)
                    {
                        const float4 e = src[q4 * kWave + lane];
                        r[4 * q4] = __builtin_fmaf(w[x], e.x, r[4 * q4]);
                        r[4 * q4 + 1] = __builtin_fmaf(w[x], e.y, r[4 * q4 + 1]);
                        r[4 * q4 + 2] = __builtin_fmaf(w[x], e.z, r[4 * q4 + 2]);
                        r[4 * q4 + 3] = __builtin_fmaf(w[x], e.w, r[4 * q4 + 3]);
                    }
                }
                if (col_ok)
                    store_dims(a, split, sp, row, dt, lg, r, inv);
            }
            if (split && col_ok && lg == 0 && kw == 0)
                store_ml(a, sp, row, mx, lsum);
        }

        // ---- the matrix-core kernel ---------------------------------------------

        // G is the group size Hq / Hkv, or 0 for a group size taken from the
        // arguments at run time.  The S * G columns of one (batch, KV head),
        // (position, head) pairs in position-major order, go 32 to a wave and
        // 32 * CW to a block; for a G that divides 32 a wave thus holds 32 / G
        // whole positions, otherwise a position's heads may straddle two waves or
        // blocks.  The block's KW groups of CW waves hold the same columns and
        // take the key tiles (32 HH keys) in turn: group kw tiles kw, kw + KW, ...
        // Their partial results meet in LDS at the end.  A wave's step is a chain
        // (its MFMAs, then the softmax, the load wait, the barrier: 1.5 us a 64-key
        // tile alone on a CU), so a launch of few blocks is as long as its longest
        // chain; groups cut the chain without the global write and read of split
        // keys (512 tokens of 32 / 8 heads: 27 us with split keys, 17.7 whole, 13.0
        // with four groups; 2048 of 16 / 8: 61, 52, 39).
        template <int G, int CW, int KW, int HH>
        __global__ __launch_bounds__(CW *KW *kWave) void attn_mfma_kernel(AttnArgs a)
        {
            const int g = G > 0 ? G : a.Hq / a.Hkv;
            constexpr int kBlockCols = 32 * CW;
            constexpr int kKeys = 32 * HH;                     // keys of a tile
            constexpr int kTileBytes = kKeys * kRowBytes;      // the K (or V) rows of a tile
            // K and V tiles, two buffers each.  Tile t's P V product is issued in
            // the step after tile t's, beside the next tile's softmax, so a V tile
            // stays resident one step longer than its K tile; V of the next step
            // is loaded into the buffer of the step before once every wave has
            // passed the barrier that ends the step.  The four buffers are separate
            // objects and the loop below names them statically, so the compiler can
            // tell that the LDS reads of a step do not depend on the loads in flight.
            __shared__ __attribute__((aligned(16))) unsigned char k_a[KW * kTileBytes];
            __shared__ __attribute__((aligned(16))) unsigned char k_b[KW * kTileBytes];
            __shared__ __attribute__((aligned(16))) unsigned char v_a[KW * kTileBytes];
            __shared__ __attribute__((aligned(16))) unsigned char v_b[KW * kTileBytes];

            const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
            const int cw = wave % CW, kw = wave / CW;
            const int lane = threadIdx.x % kWave;
            const int li = lane % 32, lg = lane / 32;

            // block -> (key slice, batch, KV head, query block).  The
            // (batch, KV head) pair runs fastest, so with a multiple of 8 pairs
            // every query block of a pair lands on one XCD (workgroups are dealt
            // to the XCDs in turn) and its L2 holds that pair's K/V; the query
            // blocks of a slice go longest first over all pairs, so that the
            // blocks that start last are the shortest (3 x 1001 tokens of 40 / 8
            // heads 54 us, 62 us with the pairs one after the other).  Slices
            // are outermost: an XCD deals its workgroups to its shader engines in
            // turn as well, and with the slice in the low bits of the id the full
            // slices of 1 x 8192 tokens (2 / 1 heads) met on half of them.
            const int pairs = static_cast<int>(gridDim.x) / (a.qblocks * a.splits);
            const int pair = static_cast<int>(blockIdx.x) % pairs;
            const int rest = static_cast<int>(blockIdx.x) / pairs;
            const int sp = rest / a.qblocks, qb = a.qblocks - 1 - rest % a.qblocks;
            const int kvh = pair % a.Hkv;
            const int64_t b = pair / a.Hkv;
            // positions, columns and key indices fit in 32 bits (checked by the
            // launcher: B * S * Hq < 2^31)
            const int32_t S = static_cast<int32_t>(a.S), start = static_cast<int32_t>(a.start);
            const int32_t n_cols = S * g;
            const int64_t block_col = static_cast<int64_t>(qb) * kBlockCols;
            const int32_t block_end = static_cast<int32_t>(block_col + kBlockCols < n_cols ? block_col + kBlockCols : n_cols);
            const int32_t s_last = (block_end - 1) / g;
            const int32_t n_keys = start + s_last + 1;
            // this block's key slice [sp * split_keys, ...) within the causal range;
            // slices past the range have nothing to do (the merge counts the same)
            const int64_t slice_begin = static_cast<int64_t>(sp) * a.split_keys;
            if (slice_begin >= n_keys)
                return;
            const int32_t k_begin = static_cast<int32_t>(slice_begin);
            const bool split = n_keys > a.split_keys;
            const int32_t k_end = n_keys - k_begin < a.split_keys ? n_keys : k_begin + a.split_keys;
            // tiles of the block [tile0, tile_end); this group's: first, first + KW, ...
            const int tile_end = (k_end + kKeys - 1) / kKeys;
            const int tile0 = k_begin / kKeys;
            const int first = tile0 + kw;
            const int steps = (tile_end - tile0 + KW - 1) / KW;
            const int mine = first < tile_end ? (tile_end - first + KW - 1) / KW : 0;

            // this lane's column
            const int64_t wave_col = block_col + 32 * cw;
            const int64_t col = wave_col + li;
            const int32_t wave_s0 = static_cast<int32_t>(wave_col / g);  // the wave's first position
            const int32_t s_col = static_cast<int32_t>(col / g);
            const int h_col = kvh * g + static_cast<int>(col % g);
            const bool col_ok = col < n_cols;
            const int32_t last_key = start + s_col;
            const bool wave_active = wave_col < n_cols;
            const bool wave_partial = wave_col + 32 > n_cols;

            const uint16_t *kbase = a.k + b * a.ks0 + kvh * a.ks2;
            const uint16_t *vbase = a.v + b * a.vs0 + kvh * a.vs2;
            const int32_t kstride = static_cast<int32_t>(a.ks1) * 2, vstride = static_cast<int32_t>(a.vs1) * 2;
            const auto kslot = [](int r, int c) __attribute__((always_inline)) { return k_slot(r, c); };
            const auto vslot = [](int r, int c) __attribute__((always_inline)) { return v_slot(r, c); };
            int32_t k_voff[Staging<CW, kKeys>::kLoads], v_voff[Staging<CW, kKeys>::kLoads];
            tile_offsets<CW, kKeys>(cw, lane, kstride, kslot, k_voff);
            tile_offsets<CW, kKeys>(cw, lane, vstride, vslot, v_voff);
            auto load_k = [&](int tile, unsigned char *buf) __attribute__((always_inline)) {
                load_tile_rows<CW, kKeys>(tile, buf + kw * kTileBytes, kbase, a.ks1, kstride, n_keys, cw, lane, k_voff,
                                          kslot);
            };
            auto load_v = [&](int tile, unsigned char *buf) __attribute__((always_inline)) {
                load_tile_rows<CW, kKeys>(tile, buf + kw * kTileBytes, vbase, a.vs1, vstride, n_keys, cw, lane, v_voff,
                                          vslot);
            };
            bf16x8_t qf[kAttD / 16];
            load_q(a, b, s_col, h_col, col_ok, lg, qf);
            int v_off[kAttD / 32];
            v_offsets(lane, v_off);
            f32x16_t o[kAttD / 32];
#pragma unroll
            for (int dt = 0; dt < kAttD / 32; ++dt)
                o[dt] = f32x16_t{};
            float m = -__builtin_huge_valf(), l = 0.0f;
            const float scale2 = a.scale * kLog2e;
            bf16x8_t phi[HH][2], plo[HH][2]; // P of the tile whose P V is still to be issued

            // One step: load K of the next tile; S^T = K(tile) Q^T; the P V of the
            // previous tile (WITH_PV); this tile's softmax; after the barrier,
            // load V of the next tile into v_prev.  (j is the step; with KW = 1
            // every group has a tile in every step.)
            auto step = [&](auto with_pv, int j, unsigned char *k_cur, unsigned char *k_next, unsigned char *v_prev)
                __attribute__((always_inline)) {
                const int tile = first + KW * j;
                if (j + 1 < mine)
                    load_k(tile + KW, k_next); // in flight while this tile is computed
                if (wave_active && (KW == 1 || j < mine))
                {
                    const int32_t key0 = tile * kKeys;
                    f32x16_t sacc[HH];
                    // The matrix phase (S = K Q^T, then the previous tile's P V)
                    // runs at raised wave priority, the softmax at the default:
                    // the other wave on the SIMD then interleaves its VALU work
                    // instead of competing for issue with the MFMAs (prefill 4%
                    // faster at config 4).
                    __builtin_amdgcn_s_setprio(1);
                    bf16x8_t vq[kAhead + 1];
                    qk_tile<HH>(k_cur + kw * kTileBytes, qf, li, lg, sacc, [&](int x) __attribute__((always_inline)) {
                        if constexpr (decltype(with_pv)::value)
                            vq[x] = read_v(v_prev + kw * kTileBytes, v_off, x);
                    });
                    if (key0 + kKeys - 1 > start + wave_s0 || wave_partial)
                        mask_tile<HH>(sacc, key0, lg, last_key, col_ok);
                    if constexpr (decltype(with_pv)::value)
                        pv_tile<HH>(v_prev + kw * kTileBytes, v_off, phi, plo, o, vq);
                    __builtin_amdgcn_s_setprio(0);
                    const float alpha = softmax_tile<HH>(sacc, scale2, m, l, phi, plo);
                    // o holds the tiles before this one at the previous reference
                    rescale(o, alpha);
                }
                // this wave's loads of the next K and this V have landed; after the
                // barrier all have, and every wave is done with this K and the V before
                __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                if (j + 1 < mine)
                    load_v(tile + KW, v_prev);
            };
            using no_pv = std::integral_constant<bool, false>;
            using with_pv = std::integral_constant<bool, true>;
            if (mine > 0)
            {
                load_k(first, k_a);
                load_v(first, v_a);
            }
            __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            // V of step j sits in v_a when j is even, else in v_b
            step(no_pv{}, 0, k_a, k_b, v_b);
            for (int j = 1; j < steps; j += 2)
            {
                step(with_pv{}, j, k_b, k_a, v_a);
                if (j + 1 < steps)
                    step(with_pv{}, j + 1, k_a, k_b, v_b);
            }
            if (wave_active && mine > 0)
            {
                const unsigned char *v_last = ((mine - 1) % 2 == 0 ? v_a : v_b) + kw * kTileBytes;
                bf16x8_t vq[kAhead + 1];
#pragma unroll
                for (int x = 0; x < kAhead; ++x)
                    vq[x] = read_v(v_last, v_off, x);
                pv_tile<HH>(v_last, v_off, phi, plo, o, vq);
            }

            const int64_t row = (b * a.S + s_col) * a.Hq + h_col;
            if constexpr (KW == 1)
            {
                store_column(a, split, sp, row, col_ok, lg, o, m, l);
            }
            else
            {
                __syncthreads(); // every wave is done with the V tiles
                merge_groups<CW, KW>(k_a, k_b, v_a, v_b, a, split, sp, row, col_ok, cw, kw, li, lg, o, m, l);
            }
        }

        // ---- few columns: decode ---------------------------------------------

        // At most 32 (position, head) columns to a (batch, KV head): one wave holds
        // them all, so the block's KW waves divide the keys, 32 at a time, and
        // share nothing until the merge.  Each wave streams its own tiles through
        // two K and two V buffers with no barrier: a buffer is refilled as soon as
        // its products are issued, and a wave waits only for the tile it needs, so
        // about 1.5 tiles of K and V (24 KiB a wave) stay in flight throughout.  What
        // bounds it is memory for many sequences (64 x 4096 keys of 32 / 8 heads: 184.9
        // us, 5.8 TB/s; 189.0 with the four-wave prefill kernel, one of whose waves
        // computed, in alternating runs) and the latency of a launch, a tile and the merge for few (1 x 8191
        // of 16 / 8: 12.2 -> 11.4 us; 40 x 3000 of 16 / 8: 119 -> 88; 19 x 8548 of
        // 5 / 1: 27 -> 18; 1 x 250: 10.0 -> 6.7).
        template <int KW>
        __global__ __launch_bounds__(KW *kWave) void attn_decode_kernel(AttnArgs a)
        {
            constexpr int kKeys = 32, kTileBytes = kKeys * kRowBytes, kL = Staging<1, kKeys>::kLoads;
            __shared__ __attribute__((aligned(16))) unsigned char k_a[KW * kTileBytes];
            __shared__ __attribute__((aligned(16))) unsigned char k_b[KW * kTileBytes];
            __shared__ __attribute__((aligned(16))) unsigned char v_a[KW * kTileBytes];
            __shared__ __attribute__((aligned(16))) unsigned char v_b[KW * kTileBytes];
            const int kw = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
            const int lane = threadIdx.x % kWave;
            const int li = lane % 32, lg = lane / 32;
            // slices of a pair side by side
            const int sp = static_cast<int>(blockIdx.x) % a.splits, pair = static_cast<int>(blockIdx.x) / a.splits;
            const int kvh = pair % a.Hkv;
            const int64_t b = pair / a.Hkv;
            const int32_t S = static_cast<int32_t>(a.S), start = static_cast<int32_t>(a.start);
            const int32_t n_keys = start + S;
            const int32_t k_begin = a.splits > 1 ? sp * a.split_keys : 0;
            const bool split = a.splits > 1;
            const int32_t k_end = split && n_keys - k_begin > a.split_keys ? k_begin + a.split_keys : n_keys;
            const int first = k_begin / kKeys + kw, tile_end = (k_end + kKeys - 1) / kKeys;
            const int mine = first < tile_end ? (tile_end - first + KW - 1) / KW : 0;

            const uint16_t *kbase = a.k + b * a.ks0 + kvh * a.ks2;
            const uint16_t *vbase = a.v + b * a.vs0 + kvh * a.vs2;
            const int32_t kstride = static_cast<int32_t>(a.ks1) * 2, vstride = static_cast<int32_t>(a.vs1) * 2;
            const auto kslot = [](int r, int c) __attribute__((always_inline)) { return k_slot(r, c); };
            const auto vslot = [](int r, int c) __attribute__((always_inline)) { return v_slot(r, c); };
            int32_t k_voff[kL], v_voff[kL];
            tile_offsets<1, kKeys>(0, lane, kstride, kslot, k_voff);
            tile_offsets<1, kKeys>(0, lane, vstride, vslot, v_voff);
            auto load_k = [&](int j, unsigned char *buf) __attribute__((always_inline)) {
                load_tile_rows<1, kKeys>(first + KW * j, buf + kw * kTileBytes, kbase, a.ks1, kstride, n_keys, 0, lane,
                                         k_voff, kslot);
            };
            auto load_v = [&](int j, unsigned char *buf) __attribute__((always_inline)) {
                load_tile_rows<1, kKeys>(first + KW * j, buf + kw * kTileBytes, vbase, a.vs1, vstride, n_keys, 0, lane,
                                         v_voff, vslot);
            };
            // the lane's column; lanes past the last one repeat a row of the last position
            const int g = a.Hq / a.Hkv;
            const int32_t s_col = li / g;
            const int h_col = kvh * g + li % g;
            const bool col_ok = s_col < S;
            bf16x8_t qf[kAttD / 16];
            load_q(a, b, s_col, h_col, col_ok, lg, qf);
            __asm__ volatile("" ::: "memory"); // Q first: waiting for it waits for no tile
            if (mine > 0)
            {
                load_k(0, k_a);
                load_v(0, v_a);
            }
            if (mine > 1)
            {
                load_k(1, k_b);
                load_v(1, v_b);
            }
            int v_off[kAttD / 32];
            v_offsets(lane, v_off);
            f32x16_t o[kAttD / 32];
#pragma unroll
            for (int dt = 0; dt < kAttD / 32; ++dt)
                o[dt] = f32x16_t{};
            float m = -__builtin_huge_valf(), l = 0.0f;
            const float scale2 = a.scale * kLog2e;

            auto step = [&](int j, unsigned char *kb, unsigned char *vb) __attribute__((always_inline)) {
                // loads by age: K(j), V(j), K(j + 1), V(j + 1)
                if (j + 1 < mine)
                    wait_loads<3 * kL>();
                else
                    wait_loads<kL>();
                f32x16_t sacc[1];
                qk_tile<1>(kb + kw * kTileBytes, qf, li, lg, sacc, [](int) __attribute__((always_inline)) {});
                wait_loads<63>();
                if (j + 2 < mine)
                    load_k(j + 2, kb);
                const int32_t key0 = (first + KW * j) * kKeys;
                if (key0 + kKeys - 1 > start)
                    mask_tile<1>(sacc, key0, lg, start + s_col, true);
                bf16x8_t phi[1][2], plo[1][2];
                const float alpha = softmax_tile<1>(sacc, scale2, m, l, phi, plo);
                rescale(o, alpha);
                // V(j), then K(j + 1), V(j + 1), K(j + 2)
                if (j + 2 < mine)
                    wait_loads<3 * kL>();
                else if (j + 1 < mine)
                    wait_loads<2 * kL>();
                else
                    wait_loads<0>();
                bf16x8_t vq[kAhead + 1];
#pragma unroll
                for (int x = 0; x < kAhead; ++x)
                    vq[x] = read_v(vb + kw * kTileBytes, v_off, x);
                pv_tile<1>(vb + kw * kTileBytes, v_off, phi, plo, o, vq);
                wait_loads<63>();
                if (j + 2 < mine)
                    load_v(j + 2, vb);
            };
            for (int j = 0; j < mine; j += 2)
            {
                step(j, k_a, v_a);
                if (j + 1 < mine)
                    step(j + 1, k_b, v_b);
            }
            const int64_t row = (b * a.S + s_col) * a.Hq + h_col;
            if constexpr (KW == 1)
                store_column(a, split, sp, row, col_ok, lg, o, m, l);
            else
            {
                __syncthreads(); // every wave is done with its tiles
                merge_groups<1, KW>(k_a, k_b, v_a, v_b, a, split, sp, row, col_ok, 0, kw, li, lg, o, m, l);
            }
        }

        // Merges the key slices of the query rows, WPR waves to a row, blocks over
        // (heads, positions, batch rows).  Every load of a round is issued before
        // any is used: lane s of each wave reads slice s's reference max and sum
        // (splits <= kMaxSplits), and wave w the unnormalised O^T of slices w,
        // w + WPR, ...  Weights 2^(m_s - max m) (the maxima are in the log2 domain),
        // then sum_s w_s O_s / sum_s w_s l_s; lane t holds dims 2t, 2t + 1, and the
        // waves' partial sums meet in LDS.
        // RANGES (more than one position): a row takes the slices its own keys
        // reach (in the others of its query block all its keys are masked), and a
        // row whose whole query block fits one slice is already done.  The slice
        // count is one 32-bit division before the loads; decode has none.
        constexpr int kMaxSplits = kAttMaxSplits;
        constexpr int kCombineWaves = 4;
        constexpr int kCombineRound = kMaxSplits / kCombineWaves; // slices whose O^T a wave loads at once
        struct CombineArgs
        {
            const float *part_o;
            const float *part_ml;
            uint16_t *out;
            int64_t rows;
            int32_t splits;
            int32_t Hq;
            int32_t S;
            int32_t start;
            int32_t split_keys;
            int32_t g;
            int32_t block_cols;
        };

        // Whether the query block of (position s, head h) fits one slice and so wrote
        // the result itself.
        __device__ __forceinline__ bool whole_block(const CombineArgs &a, int32_t s, uint32_t h)
        {
            const uint32_t g = static_cast<uint32_t>(a.g), cols = static_cast<uint32_t>(a.block_cols);
            const uint32_t col = static_cast<uint32_t>(s) * g + h % g;
            const uint32_t last = ((col / cols + 1) * cols - 1) / g; // the block's last position, before the end of S
            const int32_t s_last = last < static_cast<uint32_t>(a.S) ? static_cast<int32_t>(last) : a.S - 1;
            return a.start + s_last < a.split_keys;
        }

        template <int WPR, bool RANGES>
        __global__ __launch_bounds__(kCombineWaves * kWave) void attn_combine_kernel(CombineArgs a)
        {
            static_assert(WPR == 1 || WPR == kCombineWaves, "waves per row");
            __shared__ float2 wave_acc[kCombineWaves][kWave];
            const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
            const int lane = threadIdx.x % kWave;
            const int part = WPR == 1 ? 0 : wave;
            const int32_t h = WPR == 1 ? static_cast<int32_t>(blockIdx.x) * kCombineWaves + wave : static_cast<int32_t>(blockIdx.x);
            const int32_t s = RANGES ? static_cast<int32_t>(blockIdx.y) : 0;
            if (WPR == 1 && h >= a.Hq)
                return; // whole waves, and no barrier below
            const int64_t row = (static_cast<int64_t>(blockIdx.z) * a.S + s) * a.Hq + h;
            const int splits = RANGES ? static_cast<int>(static_cast<uint32_t>(a.start + s) / static_cast<uint32_t>(a.split_keys)) + 1
                                      : a.splits;
            float2 ml = make_float2(-__builtin_huge_valf(), 0.0f);
            if (lane < splits)
                ml = reinterpret_cast<const float2 *>(a.part_ml)[static_cast<int64_t>(lane) * a.rows + row];
            float a0 = 0.0f, a1 = 0.0f, w = 0.0f;
            auto round = [&](int s0) __attribute__((always_inline)) {
                float2 v[kCombineRound];
#pragma unroll
                for (int u = 0; u < kCombineRound; ++u)
                {
                    const int sp = s0 + part + WPR * u;
                    if (sp < splits)
                        v[u] = reinterpret_cast<const float2 *>(a.part_o + (static_cast<int64_t>(sp) * a.rows + row) *
                                                                               kAttD)[lane];
                }
                if (s0 == 0)
                {
                    float mx = ml.x;
#pragma unroll
                    for (int off = kWave / 2; off > 0; off /= 2)
                        mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
                    w = lane < splits ? __builtin_amdgcn_exp2f(ml.x - mx) : 0.0f;
                }
#pragma unroll
                for (int u = 0; u < kCombineRound; ++u)
                {
                    const int sp = s0 + part + WPR * u;
                    if (sp < splits)
                    {
                        const float ws = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), sp));
                        a0 += ws * v[u].x;
                        a1 += ws * v[u].y;
                    }
                }
            };
            round(0);
            if constexpr (WPR == 1)
                for (int s0 = kCombineRound; s0 < splits; s0 += kCombineRound)
                    round(s0);
            const float lsum = group_sum<kWave>(w * ml.y);
            bool whole = false; // the row's query block wrote the result itself
            if constexpr (RANGES)
            {
                whole = whole_block(a, s, static_cast<uint32_t>(h));
            }
            if constexpr (WPR > 1)
            {
                wave_acc[wave][lane] = make_float2(a0, a1);
                __syncthreads();
                if (part != 0)
                    return;
#pragma unroll
                for (int k = 1; k < WPR; ++k)
                {
                    a0 += wave_acc[k][lane].x;
                    a1 += wave_acc[k][lane].y;
                }
            }
            if (whole)
                return;
            const float inv = 1.0f / lsum;
            reinterpret_cast<uint32_t *>(a.out + row * kAttD)[lane] = pack_rne(a0 * inv, a1 * inv);
        }

        // The merge of many rows of few slices: 16 lanes to a row, 8 dims a lane.
        // Every lane reads its row's maxima and sums and works the weights out for
        // itself, so a wave merges four rows with no exchange between lanes (1 x 512
        // tokens after 7680, 32 / 8 heads, 16384 rows of 4 slices: 96.1 us with the
        // attention, 98.5 with a wave a row; 260 after 4096: 37.0 and 39.1).
        constexpr int kCombineFewSplits = kAttLaneMergeSplits;
        constexpr int kCombineRows = kBlock / 16; // rows of a block

        __global__ __launch_bounds__(kBlock) void attn_combine_rows_kernel(CombineArgs a)
        {
            const int64_t row = static_cast<int64_t>(blockIdx.x) * kCombineRows + threadIdx.x / 16;
            if (row >= a.rows)
                return;
            const uint32_t r = static_cast<uint32_t>(row), hq = static_cast<uint32_t>(a.Hq), S = static_cast<uint32_t>(a.S);
            const uint32_t bs = r / hq, s = bs % S;
            const int splits = static_cast<int>((static_cast<uint32_t>(a.start) + s) / static_cast<uint32_t>(a.split_keys)) + 1;
            const int d = 8 * (threadIdx.x % 16);
            float2 ml[kCombineFewSplits];
            float4 v[kCombineFewSplits][2];
#pragma unroll
            for (int i = 0; i < kCombineFewSplits; ++i)
                if (i < splits)
                {
                    const int64_t slot = static_cast<int64_t>(i) * a.rows + row;
                    ml[i] = reinterpret_cast<const float2 *>(a.part_ml)[slot];
                    const float4 *po = reinterpret_cast<const float4 *>(a.part_o + slot * kAttD + d);
                    v[i][0] = po[0];
                    v[i][1] = po[1];
                }
            float mx = -__builtin_huge_valf();
#pragma unroll
            for (int i = 0; i < kCombineFewSplits; ++i)
                if (i < splits)
                    mx = fmaxf(mx, ml[i].x);
            float acc[8] = {}, lsum = 0.0f;
#pragma unroll
            for (int i = 0; i < kCombineFewSplits; ++i)
                if (i < splits)
                {
                    const float w = __builtin_amdgcn_exp2f(ml[i].x - mx);
                    lsum += w * ml[i].y;
                    const float e[8] = {v[i][0].x, v[i][0].y, v[i][0].z, v[i][0].w, v[i][1].x, v[i][1].y, v[i][1].z, v[i][1].w};
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        acc[j] += w * e[j];
                }
            if (whole_block(a, static_cast<int32_t>(s), r % hq))
                return;
            const float inv = 1.0f / lsum;
            Vec8 out;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                out.d[j] = pack_rne(acc[2 * j] * inv, acc[2 * j + 1] * inv);
            uint2 *o = reinterpret_cast<uint2 *>(a.out + row * kAttD + d); // out is 8-byte aligned
            o[0] = make_uint2(out.d[0], out.d[1]);
            o[1] = make_uint2(out.d[2], out.d[3]);
        }

        // Generic path: one wave per query row (b, s, h); lane t holds head
        // dims t, t + 64, ... (head_dim <= 256); keys in order with the online
        // softmax of the reference.
        __global__ __launch_bounds__(kBlock) void attn_generic_kernel(AttnArgs a, int64_t rows)
        {
            const int64_t row = static_cast<int64_t>(blockIdx.x) * (kBlock / kWave) +
                                __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
            if (row >= rows)
                return;
            const int lane = threadIdx.x % kWave;
            const int h = static_cast<int>(row % a.Hq);
            const int64_t bs = row / a.Hq;
            const int64_t s = bs % a.S, b = bs / a.S;
            const int kvh = h / (a.Hq / a.Hkv);
            const int D = a.D;
            float qv[4], acc[4];
#pragma unroll
            for (int x = 0; x < 4; ++x)
            {
                const int d = lane + 64 * x;
                qv[x] = d < D ? bf_to_f(a.q[row * D + d]) : 0.0f;
                acc[x] = 0.0f;
            }
            const uint16_t *kb = a.k + b * a.ks0 + kvh * a.ks2;
            const uint16_t *vb = a.v + b * a.vs0 + kvh * a.vs2;
            float m = -__builtin_huge_valf(), l = 0.0f;
            const int64_t vis = a.start + s + 1;
            for (int64_t j = 0; j < vis; ++j)
            {
                float part = 0.0f;
#pragma unroll
                for (int x = 0; x < 4; ++x)
                {
                    const int d = lane + 64 * x;
                    if (d < D)
                        part = __builtin_fmaf(qv[x], bf_to_f(kb[j * a.ks1 + d * a.ks3]), part);
                }
                const float score = group_sum<64>(part) * a.scale;
                const float nm = fmaxf(m, score);
                const float ow = __expf(m - nm);
                const float nw = __expf(score - nm);
                l = __builtin_fmaf(l, ow, nw);
#pragma unroll
                for (int x = 0; x < 4; ++x)
                {
                    const int d = lane + 64 * x;
                    if (d < D)
                        acc[x] = __builtin_fmaf(bf_to_f(vb[j * a.vs1 + d * a.vs3]), nw, acc[x] * ow);
                }
                m = nm;
            }
#pragma unroll
            for (int x = 0; x < 4; ++x)
            {
                const int d = lane + 64 * x;
                if (d < D)
                    a.out[row * D + d] = f_to_bf(acc[x] / l);
            }
        }

        int launch_merge(const AttnArgs &a, int64_t B, int block_cols, hipStream_t stream)
        {
            if (a.splits > 1)
            {
                const CombineArgs c{a.part_o, a.part_ml, a.out, a.rows, a.splits, a.Hq, static_cast<int32_t>(a.S),
                                    static_cast<int32_t>(a.start), a.split_keys, a.Hq / a.Hkv, block_cols};
                const auto S = static_cast<unsigned>(a.S), batch = static_cast<unsigned>(B);
                const auto heads = static_cast<unsigned>(a.Hq);
                const dim3 threads(kCombineWaves * kWave);
                switch (attn_merge(a.S, a.rows, a.splits))
                {
                case AttnMerge::BlockRow:
                    if (S == 1)
                        attn_combine_kernel<kCombineWaves, false><<<dim3(heads, 1, batch), threads, 0, stream>>>(c);
                    else
                        attn_combine_kernel<kCombineWaves, true><<<dim3(heads, S, batch), threads, 0, stream>>>(c);
                    break;
                case AttnMerge::LaneRow:
                    attn_combine_rows_kernel<<<dim3(static_cast<unsigned>(blocks_for(a.rows, kCombineRows))), dim3(kBlock), 0,
                                               stream>>>(c);
                    break;
                case AttnMerge::WaveRow:
                    attn_combine_kernel<1, true>
                        <<<dim3((heads + kCombineWaves - 1) / kCombineWaves, S, batch), threads, 0, stream>>>(c);
                    break;
                }
            }
            return check_launch("grouped_query_attention");
        }

        template <int G, int CW, int KW, int HH>
        int launch_mfma(AttnArgs a, int64_t B, hipStream_t stream)
        {
            constexpr int kBlockCols = 32 * CW, kThreads = CW * KW * kWave;
            a.qblocks = static_cast<int32_t>(blocks_for(a.S * (a.Hq / a.Hkv), kBlockCols));
            const int64_t blocks = B * a.Hkv * a.qblocks * a.splits;
            // (split keys: the plan splits only grids of at most 512 blocks, so positions and
            // batch rows fit the merge's y and z dimensions)
            if (!launch_fits(blocks, kThreads) ||
                (a.splits > 1 && (a.S > 65535 || B > 65535 || !launch_fits(a.rows + B * a.S * kCombineWaves, kCombineWaves * kWave))))
                return set_error(Q3K_ERR_OVERFLOW, "GQA grid is too large");
            attn_mfma_kernel<G, CW, KW, HH><<<dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, stream>>>(a);
            return launch_merge(a, B, kBlockCols, stream);
        }

        template <int KW>
        int launch_decode(const AttnArgs &a, int64_t B, hipStream_t stream)
        {
            const int64_t blocks = B * a.Hkv * a.splits;
            if (!launch_fits(blocks, KW * kWave))
                return set_error(Q3K_ERR_OVERFLOW, "GQA grid is too large");
            attn_decode_kernel<KW><<<dim3(static_cast<unsigned>(blocks)), dim3(KW * kWave), 0, stream>>>(a);
            return launch_merge(a, B, 32, stream);
        }

        int launch_plan(const AttnArgs &a, int64_t B, const AttnPlan &plan, hipStream_t stream)
        {
            if (plan.split.decode_waves == 1)
                return launch_decode<1>(a, B, stream);
            if (plan.split.decode_waves == 2)
                return launch_decode<2>(a, B, stream);
            if (plan.split.decode_waves == 4)
                return launch_decode<4>(a, B, stream);
            if (plan.split.key_groups == 2)
                return launch_mfma<0, 4, 2, 2>(a, B, stream);
            if (plan.split.key_groups == 4)
                return launch_mfma<0, 2, 4, 1>(a, B, stream);
            switch (plan.g_instance)
            {
            case 1: return launch_mfma<1, kAttWavesPerBlock, 1, 2>(a, B, stream);
            case 2: return launch_mfma<2, kAttWavesPerBlock, 1, 2>(a, B, stream);
            case 4: return launch_mfma<4, kAttWavesPerBlock, 1, 2>(a, B, stream);
            case 8: return launch_mfma<8, kAttWavesPerBlock, 1, 2>(a, B, stream);
            case 16: return launch_mfma<16, kAttWavesPerBlock, 1, 2>(a, B, stream);
            case 32: return launch_mfma<32, kAttWavesPerBlock, 1, 2>(a, B, stream);
            default: return launch_mfma<0, kAttWavesPerBlock, 1, 2>(a, B, stream);
            }
        }
    } // namespace
} // namespace q3k

extern "C" int q3k_gqa_attention_bf16(const uint16_t *q, const uint16_t *k_cache, const uint16_t *v_cache,
                                      uint16_t *out, int64_t B, int64_t S, int32_t Hq, int32_t Hkv, int32_t D,
                                      int64_t cached, int64_t start, const int64_t *k_strides,
                                      const int64_t *v_strides, void *workspace, int64_t workspace_bytes,
                                      q3k_stream_t stream)
{
    using namespace q3k;
    if (B < 0 || S < 0)
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA batch and sequence sizes cannot be negative");
    if (Hq <= 0 || Hkv <= 0)
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA head counts must be positive");
    if (Hq % Hkv != 0)
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA query heads must be divisible by key/value heads");
    if (D <= 0 || D > 256)
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA head_dim must be between 1 and 256");
    if (start < 0)
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA start_position cannot be negative");
    if (start > cached || S != cached - start)
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA cache length must equal start_position + sequence_length");
    if (B == 0 || S == 0)
        return Q3K_OK;
    if (k_strides == nullptr || v_strides == nullptr)
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA stride arrays are null");
    for (int i = 0; i < 4; ++i)
        if (k_strides[i] < 0 || v_strides[i] < 0)
            return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA cache strides cannot be negative");
    if (q == nullptr || k_cache == nullptr || v_cache == nullptr || out == nullptr)
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA received a null pointer");
    if (!aligned_to(q, 2) || !aligned_to(k_cache, 2) || !aligned_to(v_cache, 2) || !aligned_to(out, 2))
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "GQA pointers must be 2-byte aligned");
    if (S > INT64_MAX / B || B * S > INT64_MAX / Hq || B * S * Hq > INT32_MAX)
        return set_error(Q3K_ERR_OVERFLOW, "GQA grid is too large");

    const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    AttnArgs a{q,
               k_cache,
               v_cache,
               out,
               S,
               start,
               k_strides[0],
               k_strides[1],
               k_strides[2],
               k_strides[3],
               v_strides[0],
               v_strides[1],
               v_strides[2],
               v_strides[3],
               Hq,
               Hkv,
               D,
               0,
               1.0f / __builtin_sqrtf(static_cast<float>(D)),
               1,
               INT32_MAX,
               nullptr,
               nullptr,
               B * S * Hq};
    const AttnPlan plan =
        plan_attention(B, S, Hq, Hkv, D, start, k_strides, v_strides,
                       aligned16(q) && aligned16(k_cache) && aligned16(v_cache) && aligned_to(out, 8),
                       workspace_bytes, workspace != nullptr && aligned16(workspace));
    if (plan.mfma)
    {
        if (plan.split.splits > 1)
        {
            a.splits = plan.split.splits;
            a.split_keys = plan.split.split_keys;
            a.part_o = static_cast<float *>(workspace);
            a.part_ml = a.part_o + static_cast<int64_t>(plan.split.splits) * a.rows * kAttD;
        }
        return launch_plan(a, B, plan, s);
    }
    const int64_t rows = B * S * Hq;
    const int64_t blocks = blocks_for(rows, kBlock / kWave);
    if (!launch_fits(blocks, kBlock))
        return set_error(Q3K_ERR_OVERFLOW, "GQA grid is too large");
    attn_generic_kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, s>>>(a, rows);
    return check_launch("grouped_query_attention (generic)");
}

extern "C" int64_t q3k_gqa_attention_workspace_bytes(int64_t B, int64_t S, int32_t Hq, int32_t Hkv, int32_t D,
                                                     int64_t cached)
{
    if (B <= 0 || S <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || D != q3k::kAttD || cached < S ||
        B * S * Hq > INT32_MAX)
        return 0;
    return q3k::attention_workspace_bytes(B, S, Hq, Hkv, cached);
}
