// Latent attention: tg_latent.h.

#include "tg_latent.h"

namespace {

// ---- one token -------------------------------------------------------------------------------------------------------------
// A workgroup of 16 waves takes one part of the keys for 16 heads, tile by tile of ST keys.  Scores: wave = 16 keys and a slice of
// the row; the keys come from memory in operand order (lane = key, 16 bytes of its row), queries and the new token's row
// through LDS.  The loaded pieces then go to LDS for the value sum, a product of the probabilities
// [16 heads x ST keys] (in the bf16 format two planes, value and remainder) with the tile, wave = column tiles; wider rows take
// several workgroups (blockIdx.z).  In between four waves do the softmax, a row of 16 lanes per head.
// The launch has few workgroups and is a chain of dependent stages: arguments, position, one round trip to memory, three stages
// behind barriers.  What bounds it beside these latencies is bytes through the unit's L1 (64 a clock: a query row loaded by every
// wave for itself, 147 KB a workgroup, took 2,300 clocks) and a wave's own issue (four waves that divided a linear index to find a
// piece's row took 7,600 to 15,700 clocks in front of the first product).  Against four waves and tiles of 32 keys whose scores
// came from LDS: 1000 keys, 4 heads, rows of 256 bytes 8.2 -> 5.2 us and no fold (3.0); 8 heads, rows of 640 bytes in bf16 11.9 ->
// 7.4; 4 heads, rows of 640 bytes in fp32 11.0 -> 7.1; a key group of 96 in fp32 8.0 -> 5.9.  Sixteen waves in the softmax are not
// faster than four (1,450 and 1,060 clocks): there it is the issue of their 16 rows of 64 lanes.
template <int ST>
constexpr int ST_SLICES = 256 / ST;  // of the rows in the scores
constexpr size_t ST_WIDE_LDS = 136 * 1024;  // tiles of 64 keys: LDS beside the static 22 KiB

template <class TR>
size_t latent_step_lds(int rankp, int rotp, int keys) {  // tile | queries, of wide rows their rotated parts | the new token's row
	const size_t value = (size_t)rankp * sizeof(typename TR::T), rot = (size_t)rotp * sizeof(typename TR::T);
	return (size_t)keys * (value + 16) + 16 * ((keys == 64 ? value : 0) + rot + 16) + value + rot;
}

// Element i of a rotated vector: itself, turned with its partner.
struct Turn {
	int other, pair;
	bool turns, second;
	__device__ __forceinline__ Turn(int i, int dims, int half_layout) {
		const int hd = dims / 2;
		turns = i < dims;
		second = half_layout ? i >= hd : (i & 1) != 0;
		pair = !turns ? 0 : (half_layout ? (second ? i - hd : i) : i >> 1);
		other = !turns ? i : (half_layout ? (second ? i - hd : i + hd) : i ^ 1);
	}
	__device__ __forceinline__ float operator()(float v, float o, float2 t) const {
		return turns ? fmaf(v, t.x, second ? o * t.y : -(o * t.y)) : v;
	}
};
template <class V>
__device__ __forceinline__ float rotated(const V *x, int i, const float2 *turn, int dims, int half_layout) {
	const Turn r(i, dims, half_layout);
	return r((float)x[i], (float)x[r.other], turn[r.pair]);
}
// MF: pieces of 64 bytes of a row per wave; NC: column tiles of the value part per wave (16 NC tiles of 16 per workgroup).
template <class TR, bool ROT, int ST, int MF, int NC>
__global__ __launch_bounds__(1024) void latent_step_kernel(const float *q_rows, const void *cache_rows, const int *ctr, const float *kv_rows, int host_pos, int chunk,
                                                           int window, int heads, int sizes, int key_bytes, TgLatentStep a) {
	if (tg_touch<1024>(a.touch)) return;
	typedef typename TR::T T;
	typedef typename TR::Frag Frag;
	constexpr int NS = ST_SLICES<ST>, KT = ST / 16, PLANES = TR::DT == TG_DT_BF16 ? 2 : 1, ROW = 64;
	constexpr bool SHARE = ST == 64;  // queries meet in LDS: every wave's own copies would be 16 times their bytes through the unit's L1
	extern __shared__ __align__(16) unsigned char smem[];
	const int rankp = sizes & 0xffff, rotp = ROT ? sizes >> 16 : 0;
	const int pitch = rankp * (int)sizeof(T) + 16, q0 = SHARE ? 0 : rankp, qpitch = (rankp + rotp - q0) * (int)sizeof(T) + 16;
	unsigned char *s_c = smem, *s_q = s_c + ST * pitch, *s_new = s_q + 16 * qpitch;  // s_q: [16][qpitch], rows from element q0 on
	__shared__ __align__(16) float s_part[NS][16][ST + 4];
	__shared__ __align__(16) T s_p[PLANES][16][ST + TR::KV];
	__shared__ float s_corr[16];
	const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
	// (read as a scalar: the wave's addresses depend on it)
	const int pos = host_pos >= 0 ? host_pos : *(const __attribute__((address_space(4))) int *)(unsigned long long)ctr;
	int grp = blockIdx.y, hb = 0, blocks = 1;
	if (heads > 16) {
		blocks = (heads + 15) / 16;
		grp = (int)blockIdx.y / blocks;
		hb = (int)blockIdx.y - grp * blocks;
	}
	const int g0 = grp * heads, nh = min(heads - hb * 16, 16);
	const int kfr = (rankp + rotp) / TR::KF, kfv = rankp / TR::KF, kh = (kfr + NS - 1) / NS, slice = w / KT, kt16 = 16 * (w % KT);
	const int kf_lo = min(slice * kh, kfr), nf = min(kfr - kf_lo, kh);  // (at most MF)

	// the queries; no address of them needs the position.  SHARE: wave = head, 4 elements per lane and round; else in operand order
	const float *q = q_rows + (size_t)(g0 + hb * 16 + min(SHARE ? w : lr, nh - 1)) * a.q_stride + (SHARE ? 4 * lane : lg * TR::KV);
	f32x4_t q4 = {0, 0, 0, 0};
	Frag qf[MF];
	if constexpr (SHARE) {
		if (w < nh && 4 * lane < rankp) q4 = tg_load4(q);
	} else {
#pragma unroll
		for (int i = 0; i < MF; i++) {
			if (i >= nf || kf_lo + i >= kfv) break;
#pragma unroll
			for (int e = 0; e < TR::KV / 4; e++) {
				const f32x4_t v = tg_load4(q + (kf_lo + i) * TR::KF + 4 * e);
#pragma unroll
				for (int c = 0; c < 4; c++) qf[i][4 * e + c] = (T)(lr >= nh || (ROT && (kf_lo + i) * TR::KF + lg * TR::KV + 4 * e + c < a.q_zero) ? 0.0f : v[c]);
			}
		}
	}
	const int ctx = pos + 1, lo = max(0, ctx - window), part = blockIdx.x, kb = lo + part * chunk, ke = min(ctx, kb + chunk);
	const bool mine = pos >= kb && pos < kb + chunk;
	unsigned char *cache = (unsigned char *)const_cast<void *>(cache_rows) + (size_t)grp * (kfr * ROW);
	// rows past the part's end repeat its last row, with probability 0; the new token's row is not in memory yet
	Frag tile[MF];
	auto request = [&](int k0) {
		const unsigned char *row = cache + (size_t)max(min(min(k0 + kt16 + lr, ke - 1), pos - 1), 0) * (size_t)key_bytes + lg * 16;
#pragma unroll
		for (int i = 0; i < MF; i++) {
			if (i >= nf) break;
			tile[i] = *reinterpret_cast<const Frag *>(row + (kf_lo + i) * ROW);
		}
	};
	if (kb < ke) request(kb);

	// Element j of a rotated part, requested in front of everything that waits.
	const float2 *turn = ROT ? a.rot.table + (size_t)pos * (a.rot.dims / 2) : nullptr;
	struct Rotated {
		float x, o;
		float2 t;
	};
	auto rot_request = [&](const float *x, int j0) {
		const int j = min(j0, a.rot_size - 1);
		const Turn r(j, a.rot.dims, a.rot.half_layout);
		return Rotated{x[j], x[r.other], turn[r.pair]};
	};
	auto rot_value = [&](const Rotated &v, int j) {
		const Turn r(min(j, a.rot_size - 1), a.rot.dims, a.rot.half_layout);
		return (T)(j < a.rot_size ? r(v.x, v.o, v.t) : 0.0f);
	};
	const float *qr = ROT ? a.qr + (size_t)(g0 + hb * 16 + min(w, nh - 1)) * a.qr_stride : nullptr;
	Rotated rq = {}, rk = {};
	float x = 0.0f, g = 1.0f, sq[4];
	const float *kv = kv_rows + (size_t)grp * a.kv_stride;
	if (mine) {
		x = kv[min(tid, a.rank - 1)];
		if (a.norm) {
			g = a.norm[min(tid, a.rank - 1)];
#pragma unroll
			for (int i = 0; i < 4; i++) sq[i] = kv[min(lane + 64 * i, a.rank - 1)];
		}
	}
	if constexpr (ROT) {
		if (mine && tid < rotp) rk = rot_request(a.kr + (size_t)grp * a.kr_stride, tid);
		if (w < nh && lane < rotp) rq = rot_request(qr, lane);
	}
	if (mine) {  // the new token's row, its latent normalised, by the workgroups whose part it ends
		T *dst = reinterpret_cast<T *>(cache + (size_t)pos * (size_t)key_bytes), *row = reinterpret_cast<T *>(s_new);
		float inv = 1.0f;
		if (a.norm) {  // (the sum by every wave for itself)
			float ss = 0.0f;
#pragma unroll
			for (int i = 0; i < 4; i++) ss = lane + 64 * i < a.rank ? fmaf(sq[i], sq[i], ss) : ss;
			for (int j = lane + 256; j < a.rank; j += 64) ss = fmaf(kv[j], kv[j], ss);
			inv = 1.0f / sqrtf(tg_wave_sum(ss) / (float)a.rank + a.eps);
		}
		for (int j = tid; j < rankp; j += 1024) {
			if (j >= 1024) {
				x = kv[min(j, a.rank - 1)];
				g = a.norm ? a.norm[min(j, a.rank - 1)] : 1.0f;
			}
			const T c = (T)(j < a.rank ? x * inv * g : 0.0f);
			row[j] = c;
			dst[j] = c;
		}
		if constexpr (ROT) {
			if (tid < rotp) {  // (rotp is at most 256)
				const T c = rot_value(rk, tid);
				row[rankp + tid] = c;
				dst[rankp + tid] = c;
			}
		}
	}
	if constexpr (SHARE) {
		for (int j = 4 * lane; j < rankp; j += 256) {
			if (j >= 256 && w < nh) q4 = tg_load4(q + (j - 4 * lane));
			if constexpr (ROT) {
#pragma unroll
				for (int c = 0; c < 4; c++)
					if (j + c < a.q_zero) q4[c] = 0.0f;
			}
			tg_store4(reinterpret_cast<T *>(s_q + w * qpitch) + j, q4);
		}
	}
	if constexpr (ROT) {
		for (int j = lane; j < rotp; j += 64) {
			if (j >= 64 && w < nh) rq = rot_request(qr, j);
			reinterpret_cast<T *>(s_q + w * qpitch)[rankp - q0 + j] = w < nh ? rot_value(rq, j) : (T)0.0f;
		}
	}
	if (SHARE || ROT || mine) tg_lds_barrier();
#pragma unroll
	for (int i = 0; i < MF; i++) {
		if (i >= nf) break;
		if (SHARE || (ROT && kf_lo + i >= kfv)) qf[i] = *reinterpret_cast<const Frag *>(s_q + lr * qpitch + (kf_lo + i) * ROW - q0 * (int)sizeof(T) + lg * 16);
	}

	const int ct0 = blockIdx.z * (16 * NC) + w, nct = rankp / 16;
	f32x4_t acc[NC];
#pragma unroll
	for (int c = 0; c < NC; c++) acc[c] = f32x4_t{0, 0, 0, 0};
	float m = -INFINITY, l = 0.0f;
	for (int k0 = kb; k0 < ke; k0 += ST) {
		if (mine && (unsigned)(pos - k0 - kt16) < 16u) {
#pragma unroll
			for (int i = 0; i < MF; i++) {
				if (i >= nf) break;
				const Frag f = *reinterpret_cast<const Frag *>(s_new + (kf_lo + i) * ROW + lg * 16);
				if (k0 + kt16 + lr == pos) tile[i] = f;
			}
		}
		f32x4_t sc = {0, 0, 0, 0};
#pragma unroll
		for (int i = 0; i < MF; i++) {
			if (i >= nf) break;
			sc = TR::mma(tile[i], qf[i], sc);
			if (kf_lo + i < kfv) *reinterpret_cast<Frag *>(s_c + (kt16 + lr) * pitch + (kf_lo + i) * ROW + lg * 16) = tile[i];
		}
		tg_store4(&s_part[slice][lr][kt16 + 4 * lg], sc);
		tg_lds_barrier();
		if (k0 + ST < ke) request(k0 + ST);
		if (w < 4) {  // heads 4 w + lg; lane lr: keys KT lr ...
			const int h = 4 * w + lg;
			typedef float vec __attribute__((ext_vector_type(KT)));
			typedef T tvec __attribute__((ext_vector_type(KT)));
			vec s = *reinterpret_cast<const vec *>(&s_part[0][h][KT * lr]), p;
#pragma unroll
			for (int i = 1; i < NS; i++) s += *reinterpret_cast<const vec *>(&s_part[i][h][KT * lr]);
			float mx = -INFINITY;
#pragma unroll
			for (int i = 0; i < KT; i++) {
				s[i] = k0 + KT * lr + i < ke ? s[i] * a.scale : -INFINITY;
				mx = fmaxf(mx, s[i]);
			}
			const float mn = fmaxf(m, tg_row16_max(mx)), f = expf(m - mn);
			float sum = 0.0f;
			tvec hi;
#pragma unroll
			for (int i = 0; i < KT; i++) {
				p[i] = expf(s[i] - mn);
				hi[i] = (T)p[i];
				sum += p[i];
			}
			*reinterpret_cast<tvec *>(&s_p[0][h][KT * lr]) = hi;
			if constexpr (PLANES == 2) {
				tvec rest;
#pragma unroll
				for (int i = 0; i < KT; i++) rest[i] = (T)(p[i] - (float)hi[i]);
				*reinterpret_cast<tvec *>(&s_p[1][h][KT * lr]) = rest;
			}
			if (lr == 0) s_corr[h] = f;
			l = l * f + tg_row16_sum(sum);
			m = mn;
		}
		tg_lds_barrier();
		if (k0 > kb) {
#pragma unroll
			for (int e = 0; e < 4; e++) {
				const float f = s_corr[4 * lg + e];
#pragma unroll
				for (int c = 0; c < NC; c++) acc[c][e] *= f;
			}
		}
		if (ct0 < nct) {
#pragma unroll
			for (int b = 0; b < ST / TR::KF; b++) {
				Frag pf[PLANES];
#pragma unroll
				for (int i = 0; i < PLANES; i++) pf[i] = *reinterpret_cast<const Frag *>(&s_p[i][lr][b * TR::KF + lg * TR::KV]);
#pragma unroll
				for (int c = 0; c < NC; c++) {
					const unsigned char *col = s_c + (b * TR::KF + lg * TR::KV) * pitch + (min(ct0 + 16 * c, nct - 1) * 16 + lr) * (int)sizeof(T);
					Frag cf;
#pragma unroll
					for (int i = 0; i < TR::KV; i++) cf[i] = *reinterpret_cast<const T *>(col + i * pitch);
#pragma unroll
					for (int i = 0; i < PLANES; i++) acc[c] = TR::mma(pf[i], cf, acc[c]);
				}
			}
		}
		if (k0 + ST < ke) tg_lds_barrier();
	}
	const int heads16 = a.groups * blocks * 16, hp = (int)blockIdx.y * 16;  // hp: this block's padded heads
	float *o = a.part_acc + ((size_t)part * heads16 + hp) * rankp;
#pragma unroll
	for (int c = 0; c < NC; c++) {
		const int ct = ct0 + 16 * c;
		if (ct < nct) {
#pragma unroll
			for (int e = 0; e < 4; e++) o[(size_t)(4 * lg + e) * rankp + ct * 16 + lr] = acc[c][e];
		}
	}
	if (blockIdx.z == 0 && w < 4 && lr == 0) *reinterpret_cast<float2 *>(a.part_ml + ((size_t)part * heads16 + hp + 4 * w + lg) * 2) = float2{m, l};
}

// groups > 0: the normalised sum of real head (group, head) instead, [groups * heads][out_stride]
__global__ __launch_bounds__(256) void latent_fold_kernel(const float *acc, const float *ml, int nb, int heads16, int rankp, float *out_acc,
                                                          float *out_ml, int groups, int heads, int out_stride) {
	__shared__ float s_f[TG_LATENT_MAX_BLOCKS];
	__shared__ float s_r[4];
	const int hp16 = (heads + 15) / 16 * 16, real = (int)blockIdx.x;
	const int h = groups ? real / heads * hp16 + real % heads : real, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
	float m = -INFINITY;
	for (int b = tid; b < nb; b += 256) m = fmaxf(m, ml[((size_t)b * heads16 + h) * 2]);
	m = tg_wave_max(m);
	if (lane == 0) s_r[w] = m;
	__syncthreads();
	m = fmaxf(fmaxf(s_r[0], s_r[1]), fmaxf(s_r[2], s_r[3]));
	__syncthreads();
	float l = 0.0f;
	for (int b = tid; b < nb; b += 256) {
		const float f = expf(ml[((size_t)b * heads16 + h) * 2] - m);
		s_f[b] = f;
		l += f * ml[((size_t)b * heads16 + h) * 2 + 1];
	}
	l = tg_wave_sum(l);
	if (lane == 0) s_r[w] = l;
	__syncthreads();
	l = (s_r[0] + s_r[1]) + (s_r[2] + s_r[3]);
	if (!groups && tid == 0 && blockIdx.y == 0) {
		out_ml[2 * h] = m;
		out_ml[2 * h + 1] = l;
	}
	const int j = blockIdx.y * 64 + lane, jc = min(j, rankp - 1);  // a wave per quarter of the parts
	float a = 0.0f;
	for (int b = w; b < nb; b += 64) {
		float v[16];
#pragma unroll
		for (int i = 0; i < 16; i++) v[i] = acc[((size_t)min(b + 4 * i, nb - 1) * heads16 + h) * rankp + jc];
#pragma unroll
		for (int i = 0; i < 16; i++) a = fmaf(b + 4 * i < nb ? s_f[min(b + 4 * i, nb - 1)] : 0.0f, v[i], a);
	}
	__shared__ float s_a[4][64];
	s_a[w][lane] = a;
	__syncthreads();
	if (w != 0 || j >= rankp) return;
	const float sum = (s_a[0][lane] + s_a[1][lane]) + (s_a[2][lane] + s_a[3][lane]);
	if (groups) out_acc[(size_t)real * out_stride + j] = sum / l;
	else out_acc[(size_t)h * rankp + j] = sum;
}

// ---- many tokens -------------------------------------------------------------------------------------------------------------
// a wave per token and group
template <class TR, class SRC>
__global__ __launch_bounds__(256) void latent_rows_kernel(TgLatentCacheRows a) {
	typedef typename TR::T T;
	const int e = blockIdx.x * 4 + (threadIdx.x >> 6), t = e / a.groups, grp = e - t * a.groups, lane = threadIdx.x & 63;
	if (t >= a.n) return;
	const SRC *x = (const SRC *)a.kv + (size_t)t * a.ld + (size_t)grp * a.kv_stride, *r = (const SRC *)a.kr + (size_t)t * a.ld + (size_t)grp * a.kr_stride;
	float inv = 1.0f;
	if (a.norm) {
		float ss = 0.0f;
		for (int j = lane; j < a.rank; j += 64) ss = fmaf((float)x[j], (float)x[j], ss);
		ss = tg_wave_sum(ss);
		inv = 1.0f / sqrtf(ss / (float)a.rank + a.eps);
	}
	const int pos = a.past + t;
	T *row = (T *)a.cache + ((size_t)pos * a.groups + grp) * (a.rankp + a.rotp);
	for (int j = lane; j < a.rankp; j += 64) {
		const int jc = j < a.rank ? j : 0;
		const float c = (float)x[jc] * inv * (a.norm ? a.norm[jc] : 1.0f);
		row[j] = (T)(j < a.rank ? c : 0.0f);
	}
	const float2 *turn = a.rot.table + (size_t)pos * (a.rot.dims / 2);
	for (int j = lane; j < a.rotp; j += 64) row[a.rankp + j] = (T)(j < a.rot_size ? rotated(r, j, turn, a.rot.dims, a.rot.half_layout) : 0.0f);
}

// a lane per pair
template <class T>
__global__ __launch_bounds__(256) void rot_rows_kernel(T *rows, int ld, int past, int first, int count, int stride, TgRot rot) {
	const int hd = rot.dims / 2, per = count * hd, t = blockIdx.y;
	const int e = blockIdx.x * 256 + threadIdx.x;
	if (e >= per) return;
	const int v = e / hd, i = e - v * hd;
	T *x = rows + (size_t)t * ld + first + (size_t)v * stride;
	T *p = x + (rot.half_layout ? i : 2 * i), *q = x + (rot.half_layout ? i + hd : 2 * i + 1);
	const float2 c = rot.table[(size_t)(past + t) * hd + i];
	const float u = (float)*p, w = (float)*q;
	*p = (T)fmaf(u, c.x, -(w * c.y));
	*q = (T)fmaf(w, c.x, u * c.y);
}

// 64 keys x 32 dimensions of a group per workgroup: rotated keys straight through, values transposed through LDS into the
// key order of the attention operand; keys past the end are zero values
template <class TR>
__global__ __launch_bounds__(256) void key_values_kernel(TgKeyValues a) {
	typedef typename TR::T T;
	__shared__ T s_v[32][64 + 4];
	const int grp = blockIdx.y, d0 = blockIdx.z * 32, k0 = blockIdx.x * 64, tid = threadIdx.x;
	const int rowp = a.dimp + a.rotp;
	for (int e = tid; e < 64 * 32; e += 256) {
		const int kk = e >> 5, d = e & 31, key = k0 + kk;
		T v = (T)0.0f;
		if (key < a.n) {
			const T *row = (const T *)a.cache + ((size_t)(a.lo + key) * a.groups + grp) * rowp;
			v = row[d0 + d];
			((T *)a.k)[(size_t)key * a.groups * a.dimp + (size_t)grp * a.dimp + d0 + d] = d0 + d < a.rot_size ? row[a.dimp + d0 + d] : v;
		}
		int at = kk;
		if constexpr (TR::DT == TG_DT_BF16) at = (kk & 32) + 8 * ((kk & 15) >> 2) + 4 * ((kk >> 4) & 1) + (kk & 3);
		s_v[d][at] = v;
	}
	__syncthreads();
	for (int e = tid; e < 64 * 32; e += 256) {
		const int d = e >> 6, at = e & 63;
		((T *)a.vt)[(size_t)(grp * a.dimp + d0 + d) * a.ldv + k0 + at] = s_v[d][at];
	}
}

// A workgroup: one head, 64 QT queries (wave: 16 QT of them).  Per tile of KT keys: K and V^T fragments go global ->
// registers -> LDS, the next tile's loads in flight during this one's arithmetic.  Scores are taken as K Q^T, so a lane holds
// four consecutive keys of one query and the probabilities are already the second operand of V^T P^T; in the bf16 format they
// enter it as two bf16 planes (value and remainder).
// Sizes are compile-time buckets (DM >= dimp, VM >= vdimp): query elements past the head are zero, value rows past it are
// computed from repeated rows and not stored, so that no branch stands between the LDS reads and matrix instructions.
// WIDE: with a window, a rotated part or grouped heads.
template <class TR, int DM, int VM, int KT, int QT, bool WIDE>
__global__ __launch_bounds__(256, 2) void latent_attn_kernel(TgLatentRows a) {
	typedef typename TR::T T;
	typedef typename TR::Frag Frag;
	constexpr int ND = DM / TR::KF, NV = VM / 16, NK = KT / 16, NB = KT / TR::KF;
	constexpr int KFRAGS = NK * ND, NF = KFRAGS + NV * NB, PW = NF / 4;
	static_assert(NF % 4 == 0 && NB >= 1, "");
	__shared__ __align__(16) Frag lds[NF * 64];
	const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lg = lane >> 4;
	// Query tiles from both ends: the first half of the launch takes the long rows, longest first, the second half the
	// short ones, shortest first, so that the workgroups that meet on a compute unit have about the same work together.
	const int nqt = (int)gridDim.y, y = (int)blockIdx.y, half = (nqt + 1) / 2;
	const int h = blockIdx.x, kh = WIDE ? h / a.group : h, qb = (y < half ? nqt - 1 - y : y - half) * 64 * QT;
	const int kn = a.dimp / TR::KF, kd = (a.dimp + (WIDE ? a.rotp : 0)) / TR::KF, nv = a.vdimp / 16;
	const T *Q = (const T *)a.q, *K = (const T *)a.k + (size_t)kh * a.dimp, *V = (const T *)a.vt + (size_t)kh * a.vdimp * a.ldv;
	const T *R = (const T *)a.kr;
	const float sl2 = fabsf(a.scale) * 1.44269504088896340736f;  // (the sign goes to the queries: maxima are taken before scaling)
	const bool neg = a.scale < 0.0f;

	Frag qf[QT][ND];
	int qi[QT];
#pragma unroll
	for (int s = 0; s < QT; s++) {
		qi[s] = qb + w * 16 * QT + s * 16 + lr;
		const T *row = Q + (size_t)min(qi[s], a.n - 1) * a.ldq + (size_t)h * (a.dimp + (WIDE ? a.rotp : 0)) + lg * TR::KV;
#pragma unroll
		for (int d = 0; d < ND; d++) {
			qf[s][d] = *reinterpret_cast<const Frag *>(row + (d < kd ? d : 0) * TR::KF);
			if (d >= kd) qf[s][d] = Frag{};
			if (neg) qf[s][d] = -qf[s][d];
		}
	}
	f32x4_t o[QT][NV];
	float m[QT], l[QT];
#pragma unroll
	for (int s = 0; s < QT; s++) {
		m[s] = -1e30f;  // below every score; finite, so that a tile without a visible key leaves everything as it is
		l[s] = 0.0f;
#pragma unroll
		for (int v = 0; v < NV; v++) o[s][v] = f32x4_t{0, 0, 0, 0};
	}
	const int last = a.past + min(qb + 64 * QT, a.n) - 1;  // the last key any of these queries sees
	const int nt = last / KT + 1, ctx = a.past + a.n, tb = WIDE ? max(a.past + qb - a.window + 1, 0) / KT : 0;
	Frag st[PW];
	auto fetch = [&](int k0) {
#pragma unroll
		for (int i = 0; i < PW; i++) {
			const int f = i * 4 + w;
			const T *p;
			if (f < KFRAGS) {
				const int kt = f / ND, d = f % ND;
				const size_t key = (size_t)min(k0 + kt * 16 + lr, ctx - 1);
				if constexpr (!WIDE) p = K + key * a.ldk + (d < kd ? d : 0) * TR::KF + lg * TR::KV;
				else p = (d < kn || d >= kd ? K + key * a.ldk + (d < kn ? d : 0) * TR::KF : R + key * a.ldkr + (d - kn) * TR::KF) + lg * TR::KV;
			} else {
				const int v = (f - KFRAGS) / NB, b = (f - KFRAGS) % NB;
				p = V + (size_t)((v < nv ? v : 0) * 16 + lr) * a.ldv + k0 + b * TR::KF + lg * TR::KV;
			}
			st[i] = *reinterpret_cast<const Frag *>(p);
		}
	};
	auto put = [&]() {
#pragma unroll
		for (int i = 0; i < PW; i++) lds[(i * 4 + w) * 64 + lane] = st[i];
	};
	fetch(tb * KT);
	put();
	tg_lds_barrier();
	for (int t = tb; t < nt; t++) {
		const int k0 = t * KT;
		fetch((t + 1 < nt ? t + 1 : t) * KT);
		f32x4_t sc[QT][NK];
#pragma unroll
		for (int kt = 0; kt < NK; kt++) {
#pragma unroll
			for (int s = 0; s < QT; s++) sc[s][kt] = f32x4_t{0, 0, 0, 0};
#pragma unroll
			for (int d = 0; d < ND; d++) {
				const Frag kf = lds[(kt * ND + d) * 64 + lane];
#pragma unroll
				for (int s = 0; s < QT; s++) sc[s][kt] = TR::mma(kf, qf[s][d], sc[s][kt]);
			}
		}
		// keys past a query only in the tiles that reach the wave's first query, keys before its window in those that do not
		// reach the last query's
		const int first_q = a.past + qb + w * 16 * QT;
		const bool masked = k0 + KT - 1 > first_q || (WIDE && k0 < first_q + 16 * QT - a.window);
#pragma unroll
		for (int s = 0; s < QT; s++) {
			if (masked) {
				const int lim = a.past + qi[s] - k0 - 4 * lg, low = WIDE ? lim - a.window : -TG_NO_WINDOW;
#pragma unroll
				for (int kt = 0; kt < NK; kt++)
#pragma unroll
					for (int e = 0; e < 4; e++) sc[s][kt][e] = kt * 16 + e <= lim && (!WIDE || kt * 16 + e > low) ? sc[s][kt][e] : -INFINITY;
			}
			float mt = -INFINITY;
#pragma unroll
			for (int kt = 0; kt < NK; kt++)
#pragma unroll
				for (int e = 0; e < 4; e++) mt = fmaxf(mt, sc[s][kt][e]);
			mt = fmaxf(mt, tg_red_partner<32>(mt));
			mt = fmaxf(mt, tg_red_partner<16>(mt));
			const float mn = fmaxf(m[s], mt * sl2);
			if (__ballot(mn > m[s])) {
				const float f = __builtin_amdgcn_exp2f(m[s] - mn);
				l[s] *= f;
#pragma unroll
				for (int v = 0; v < NV; v++)
#pragma unroll
					for (int e = 0; e < 4; e++) o[s][v][e] *= f;
				m[s] = mn;
			}
			float sum = 0.0f;
#pragma unroll
			for (int kt = 0; kt < NK; kt++)
#pragma unroll
				for (int e = 0; e < 4; e++) {
					const float p = __builtin_amdgcn_exp2f(fmaf(sc[s][kt][e], sl2, -mn));
					sc[s][kt][e] = p;
					sum += p;
				}
			l[s] += sum;
		}
#pragma unroll
		for (int b = 0; b < NB; b++) {
			Frag ph[QT], pl[QT];
#pragma unroll
			for (int s = 0; s < QT; s++) {
				if constexpr (TR::DT == TG_DT_BF16) {
#pragma unroll
					for (int e = 0; e < 8; e++) {
						const float p = sc[s][2 * b + (e >> 2)][e & 3];
						const __bf16 hi = (__bf16)p;
						ph[s][e] = hi;
						pl[s][e] = (__bf16)(p - (float)hi);
					}
				} else {
					ph[s] = sc[s][b];
				}
			}
#pragma unroll
			for (int v = 0; v < NV; v++) {
				const Frag vf = lds[(KFRAGS + v * NB + b) * 64 + lane];
#pragma unroll
				for (int s = 0; s < QT; s++) {
					o[s][v] = TR::mma(vf, ph[s], o[s][v]);
					if constexpr (TR::DT == TG_DT_BF16) o[s][v] = TR::mma(vf, pl[s], o[s][v]);
				}
			}
		}
		tg_lds_barrier();
		put();
		tg_lds_barrier();
	}
#pragma unroll
	for (int s = 0; s < QT; s++) {
		float ls = l[s];
		ls += tg_red_partner<32>(ls);
		ls += tg_red_partner<16>(ls);
		if (qi[s] >= a.n) continue;
		const float f = (a.gate ? tg_sigmoid(a.gate[(size_t)qi[s] * a.ld_gate + h]) : 1.0f) / ls;
		T *dst = (T *)a.out + (size_t)qi[s] * a.ldo + (size_t)h * a.vdimp + 4 * lg;
#pragma unroll
		for (int v = 0; v < NV; v++)
			if (v < nv) {
				f32x4_t r;
#pragma unroll
				for (int e = 0; e < 4; e++) r[e] = o[s][v][e] * f;
				tg_store4(dst + v * 16, r);
			}
		if (h == a.heads - 1)
			for (int c = a.heads * a.vdimp + 4 * lg; c < a.ldo; c += 16) tg_store4((T *)a.out + (size_t)qi[s] * a.ldo + c, f32x4_t{0, 0, 0, 0});
	}
}

template <class TR, int DM, int VM, int KT, bool WIDE>
void launch_bucket_w(const TgLatentRows &a, hipStream_t s) {
	// 128-query tiles (half the LDS reads per product) where they fill the device twice
	if constexpr (TR::DT == TG_DT_BF16 && DM <= 128 && VM <= 128) {
		if (a.heads * ((a.n + 127) / 128) >= 512) {
			hipLaunchKernelGGL((latent_attn_kernel<TR, DM, VM, KT, 2, WIDE>), dim3((unsigned)a.heads, (unsigned)((a.n + 127) / 128)), dim3(256), 0, s, a);
			return;
		}
	}
	hipLaunchKernelGGL((latent_attn_kernel<TR, DM, VM, KT, 1, WIDE>), dim3((unsigned)a.heads, (unsigned)((a.n + 63) / 64)), dim3(256), 0, s, a);
}
template <class TR, int DM, int VM, int KT>
void launch_bucket(const TgLatentRows &a, hipStream_t s) {
	if (a.rotp || a.group > 1 || a.window < TG_NO_WINDOW) launch_bucket_w<TR, DM, VM, KT, true>(a, s);
	else launch_bucket_w<TR, DM, VM, KT, false>(a, s);
}

template <class TR>
void launch_attention(const TgLatentRows &a, hipStream_t s) {
	constexpr int W = TR::DT == TG_DT_BF16 ? 64 : 32;  // keys per tile of the wide buckets
	const int d = a.dimp + a.rotp, v = a.vdimp;
	if (d <= 64 && v <= 64) launch_bucket<TR, 64, 64, 64>(a, s);
	else if (d <= 64 && v <= 128) launch_bucket<TR, 64, 128, 64>(a, s);
	else if (d <= 128 && v <= 64) launch_bucket<TR, 128, 64, 64>(a, s);
	else if (d <= 128 && v <= 128) launch_bucket<TR, 128, 128, W>(a, s);
	else if (d <= 192 && v <= 128) launch_bucket<TR, 192, 128, 32>(a, s);
	else launch_bucket<TR, 256, 256, 32>(a, s);
}

}  // namespace

namespace {
template <class TR>
void launch_step(const TgLatentStep &a, hipStream_t s) {
	TgLatentStep t = a;
	const dim3 grid = tg_touch_grid(dim3((unsigned)a.nb, (unsigned)(a.groups * ((a.heads + 15) / 16)), (unsigned)((a.rankp + 511) / 512)), &t.touch, a.touch_blocks);
	auto go = [&](auto *kernel, size_t lds) {
		if (lds > 40 * 1024) (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
		hipLaunchKernelGGL(kernel, grid, dim3(1024), lds, s, a.q, a.cache, a.ctr, a.kv, a.host_pos, a.chunk, a.window, a.heads, a.rankp | a.rotp << 16,
		                   a.groups * a.rowp() * (int)sizeof(typename TR::T), t);
	};
	// tiles of 64 keys wherever they fit, 32 for wider rows; rows of more than 768 bytes take more pieces per wave
	const size_t wide = latent_step_lds<TR>(a.rankp, a.rotp, 64), narrow = latent_step_lds<TR>(a.rankp, a.rotp, 32);
	const size_t row = (size_t)a.rowp() * sizeof(typename TR::T);
	if (row > 2048 || wide > ST_WIDE_LDS) {
		if (a.rotp) go(latent_step_kernel<TR, true, 32, 7, 2>, narrow);
		else go(latent_step_kernel<TR, false, 32, 7, 2>, narrow);
	} else if (row <= 768 && a.rankp <= 256) {
		if (a.rotp) go(latent_step_kernel<TR, true, 64, 3, 1>, wide);
		else go(latent_step_kernel<TR, false, 64, 3, 1>, wide);
	} else {
		if (a.rotp) go(latent_step_kernel<TR, true, 64, 8, 2>, wide);
		else go(latent_step_kernel<TR, false, 64, 8, 2>, wide);
	}
}
}  // namespace

void tg_launch_latent_step(const TgLatentStep &a, int dt, hipStream_t s) {
	if (dt == TG_DT_BF16) launch_step<TgB16>(a, s);
	else launch_step<TgF32>(a, s);
}

void tg_launch_latent_fold(const float *acc, const float *ml, int nb, int heads_padded, int rankp, float *out_acc, float *out_ml, hipStream_t s) {
	hipLaunchKernelGGL(latent_fold_kernel, dim3((unsigned)heads_padded, (unsigned)((rankp + 63) / 64)), dim3(256), 0, s, acc, ml, nb, heads_padded, rankp,
	                   out_acc, out_ml, 0, 1, 0);
}

void tg_launch_latent_finish(const float *acc, const float *ml, int nb, int groups, int heads, int rankp, float *out, int out_stride, hipStream_t s) {
	hipLaunchKernelGGL(latent_fold_kernel, dim3((unsigned)(groups * heads), (unsigned)((rankp + 63) / 64)), dim3(256), 0, s, acc, ml, nb,
	                   groups * tg_up(heads, 16), rankp, out, (float *)nullptr, groups, heads, out_stride);
}

namespace {
template <class TR>
void launch_cache_rows(const TgLatentCacheRows &a, hipStream_t s) {
	const dim3 grid((unsigned)((a.n * a.groups + 3) / 4));
	if (a.f32) hipLaunchKernelGGL((latent_rows_kernel<TR, float>), grid, dim3(256), 0, s, a);
	else hipLaunchKernelGGL((latent_rows_kernel<TR, typename TR::T>), grid, dim3(256), 0, s, a);
}
}  // namespace

void tg_launch_latent_rows(const TgLatentCacheRows &a, int dt, hipStream_t s) {
	if (dt == TG_DT_BF16) launch_cache_rows<TgB16>(a, s);
	else launch_cache_rows<TgF32>(a, s);
}

void tg_launch_rot_rows(void *rows, int ld, int n, int past, int first, int count, int stride, const TgRot &rot, int dt, hipStream_t s) {
	const dim3 grid((unsigned)((count * (rot.dims / 2) + 255) / 256), (unsigned)n);
	if (dt == TG_DT_BF16) hipLaunchKernelGGL((rot_rows_kernel<__bf16>), grid, dim3(256), 0, s, (__bf16 *)rows, ld, past, first, count, stride, rot);
	else hipLaunchKernelGGL((rot_rows_kernel<float>), grid, dim3(256), 0, s, (float *)rows, ld, past, first, count, stride, rot);
}

void tg_launch_key_values(const TgKeyValues &a, int dt, hipStream_t s) {
	const dim3 grid((unsigned)((a.n + 63) / 64), (unsigned)a.groups, (unsigned)(a.dimp / 32));
	if (dt == TG_DT_BF16) hipLaunchKernelGGL((key_values_kernel<TgB16>), grid, dim3(256), 0, s, a);
	else hipLaunchKernelGGL((key_values_kernel<TgF32>), grid, dim3(256), 0, s, a);
}

void tg_launch_latent_attention(const TgLatentRows &a, int dt, hipStream_t s) {
	if (dt == TG_DT_BF16) launch_attention<TgB16>(a, s);
	else launch_attention<TgF32>(a, s);
}
