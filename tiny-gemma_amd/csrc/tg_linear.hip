// Products with bfloat16 or float32 weights: packing, one-row products (decode) and tiled products (prefill).
// Layout and number formats: tg_linear.h.

#include "tg_linear.h"

#include <type_traits>

namespace {

// ---- packing (load time) -----------------------------------------------------------------------------------------------
__device__ __forceinline__ float pack_read(const TgPack &p, int i, int j) {
	const int gi = i / p.gp, ri = i - gi * p.gp, gj = j / p.kgp, rj = j - gj * p.kgp;
	const int r = gi * p.g + ri, c = gj * p.kg + rj;
	if (ri >= p.g || rj >= p.kg || r >= p.rsrc || c >= p.ksrc) return 0.0f;
	const size_t at = p.transpose ? (size_t)c * p.src_ld + r : (size_t)r * p.src_ld + c;
	return (p.src_f32 ? ((const float *)p.src)[at] : (float)((const __bf16 *)p.src)[at]) + p.add;
}

template <class TR>
__global__ __launch_bounds__(256) void pack_kernel(typename TR::T *dst, int k, TgPack p) {
	const long long total = (long long)p.rows * p.cols;
	for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long long)gridDim.x * 256) {
		const int i = (int)(e / p.cols), j = (int)(e - (long long)i * p.cols);
		const int row = (i / 16) * 16 * p.frag_step + p.frag_off * 16 + i % 16;
		const size_t frag = (size_t)(row / 16) * (k / TR::KF) + j / TR::KF;
		const int lane = row % 16 + 16 * ((j % TR::KF) / TR::KV);
		dst[frag * 64 * TR::KV + lane * TR::KV + j % TR::KV] = (typename TR::T)pack_read(p, i, j);
	}
}

__global__ __launch_bounds__(256) void unpack_f32_kernel(float *dst, int ld, TgPack p) {
	const long long total = (long long)p.rows * p.cols;
	for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long long)gridDim.x * 256) {
		const int i = (int)(e / p.cols), j = (int)(e - (long long)i * p.cols);
		dst[(size_t)i * ld + j] = pack_read(p, i, j);
	}
}

// ---- one-row products ----------------------------------------------------------------------------------------------------
constexpr int NT = 256;
template <int N>
using Const = std::integral_constant<int, N>;

// Experts by rank: expert e is chosen when fewer than `top` experts have a larger choice score (or the same one and a
// lower index).  s_sel / s_val (LDS, top entries): the chosen experts in rank order and their scores.
__device__ __forceinline__ void choose_experts(const float *logits, const float *correction, int E, int top, float *s_choice, int *s_sel,
                                               float *s_val) {
	const int E4 = (E + 3) & ~3;  // s_choice has room for a multiple of four
	for (int e = threadIdx.x; e < E4; e += NT) s_choice[e] = e < E ? tg_choice_score(tg_sigmoid(logits[e]), correction[e]) : -INFINITY;
	__syncthreads();
	for (int e = threadIdx.x; e < E; e += NT) {
		const float c = s_choice[e];
		int rank = 0;
		for (int o = 0; o < E4; o += 4) {
			const f32x4_t co = tg_load4(s_choice + o);
#pragma unroll
			for (int i = 0; i < 4; i++) rank += (co[i] > c || (co[i] == c && o + i < e)) ? 1 : 0;
		}
		if (rank < top) {
			s_sel[rank] = e;
			s_val[rank] = tg_sigmoid(logits[e]);
		}
	}
	__syncthreads();
}

// A launch is a chain of dependent memory round trips, so every prologue requests all of its inputs before it uses one
// (clamped indices, no loads under branches), and the first round of the weight stream right behind them: waits are in
// order, the prologue's arithmetic then runs while the weights are on their way.
//
// The same goes for the arguments.  Read from the descriptor field by field where they are used, they were five scalar round
// trips in front of the first vector load.  What the first loads need are therefore leading arguments of the kernel, which the
// dispatcher preloads into scalar registers (VecHot; 14 dwords), and the rest of the descriptor is fetched in one batch behind
// those loads (fetch_rest).

// v, or +0 where a duplicate of the last part was loaded for an even count: a mask and no condition, behind which the compiler
// would move the load, with a wait of its own
__device__ __forceinline__ float masked(float v, bool is) { return __uint_as_float(__float_as_uint(v) & (is ? ~0u : 0u)); }

struct VecHot {
	const void *a[4];
	int i[6];
};
constexpr size_t VEC_DESC_OFFSET = sizeof(VecHot);  // of the descriptor in the argument block
static_assert(VEC_DESC_OFFSET % alignof(TgVec) == 0 && sizeof(VecHot) == 56, "leading arguments of vec_kernel");

template <int PRO, int EPI>
VecHot vec_hot(const TgVec &v) {
	VecHot h = {{v.x, nullptr, nullptr, nullptr}, {v.kfrags, v.ksplit, 0, 0, 0, 0}};
	if (PRO == TG_VP_DYT || PRO == TG_VP_ROUTE || PRO == TG_VP_RMS) {
		h = VecHot{{v.embed ? v.embed : v.x, v.nw, PRO == TG_VP_RMS ? v.post : v.nb, v.pend}, {v.kfrags, v.ksplit, v.nparts, v.pend_stride, v.embed ? 1 : 0, 0}};
	} else if (PRO == TG_VP_HEADNORM) {
		h = VecHot{{v.x, v.nw, v.gate, nullptr}, {v.kfrags, v.ksplit, v.vdimp, v.heads16, 0, 0}};
	} else if (PRO == TG_VP_MERGE || PRO == TG_VP_MERGE_HEADS) {
		h = VecHot{{v.part_acc, v.part_ml, nullptr, nullptr}, {v.kfrags, v.ksplit, v.nmerge, v.heads16, v.x_zstride, v.group | v.heads << 16}};
	} else if (PRO == TG_VP_EXPERT) {
		h = VecHot{{v.x, v.logits, v.correction, nullptr}, {v.kfrags, v.ksplit, v.experts, v.top, 0, 0}};
	} else {
		h = VecHot{{v.x, EPI == TG_VE_WEIGHTED ? v.sel : nullptr, nullptr, nullptr}, {v.kfrags, v.ksplit, v.x_zstride, 0, 0, 0}};
	}
	return h;
}
template <int PRO, int EPI>
__device__ __forceinline__ TgVec with_hot(const TgVec &v, const void *a0, const void *a1, const void *a2, const void *a3, int i0, int i1, int i2, int i3, int i4,
                                          int i5) {
	TgVec p = v;
	p.kfrags = i0;
	p.ksplit = i1;
	p.x = (const float *)a0;
	if (PRO == TG_VP_DYT || PRO == TG_VP_ROUTE || PRO == TG_VP_RMS) {
		p.embed = i4 ? a0 : nullptr;
		p.embed_ld = 0;  // (read where there is a table)
		p.embed_scale = 0.0f;
		p.nw = (const float *)a1;
		p.nb = p.post = (const float *)a2;
		p.pend = (const float *)a3;
		p.nparts = i2;
		p.pend_stride = i3;
	} else if (PRO == TG_VP_HEADNORM) {
		p.nw = (const float *)a1;
		p.gate = (const float *)a2;
		p.vdimp = i2;
		p.heads16 = i3;
	} else if (PRO == TG_VP_MERGE || PRO == TG_VP_MERGE_HEADS) {
		p.part_acc = (const float *)a0;
		p.part_ml = (const float *)a1;
		p.nmerge = i2;
		p.heads16 = i3;
		p.x_zstride = i4;
		p.vdimp = PRO == TG_VP_MERGE_HEADS ? i4 : p.vdimp;
		p.group = i5 & 0xffff;
		p.heads = i5 >> 16;
	} else if (PRO == TG_VP_EXPERT) {
		p.logits = (const float *)a1;
		p.correction = (const float *)a2;
		p.experts = i2;
		p.top = i3;
	} else {
		p.x_zstride = i2;
		if (EPI == TG_VE_WEIGHTED) p.sel = (int *)a1;
	}
	return p;
}

// NTL: tiles per wave (2: a gate|up pair); KW: waves that share a tile's K (4), or 1: every wave has tiles of its own;
// U: fragments in flight per lane and tile; VP (prologues with a norm): the vector's length class, see vec_class()
template <class TR, int PRO, int EPI, int NTL, int KW, int U, int VP>
__global__ __launch_bounds__(NT) void vec_kernel(const void *a0, const void *a1, const void *a2, const void *a3, int i0, int i1, int i2, int i3, int i4,
                                                 int i5, const TgVec p_in) {
	TgVec p = with_hot<PRO, EPI>(p_in, a0, a1, a2, a3, i0, i1, i2, i3, i4, i5);
	typedef typename TR::T T;
	typedef typename TR::Frag Frag;
	extern __shared__ __align__(16) unsigned char smem[];
	T *xs = reinterpret_cast<T *>(smem);
	__shared__ float s_red[4][NTL * 16];
	__shared__ float s_misc[64];
	const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
	const int part = blockIdx.y, z = blockIdx.z;
	const int per = (p.kfrags + p.ksplit - 1) / p.ksplit;
	const int kb = part * per, ke = min(p.kfrags, kb + per), nk = max(ke - kb, 0);
	const int k0 = kb * TR::KF, kn = nk * TR::KF;

	int zw = z;
	auto choose = [&](const float *logits) {
		// LDS: choice scores [experts, padded] | selected [top] | their scores [top] behind the vector
		float *s_choice = reinterpret_cast<float *>(smem + sizeof(T) * (size_t)(per + KW * U) * TR::KF);
		int *s_sel = reinterpret_cast<int *>(s_choice + ((p.experts + 3) & ~3));
		float *s_val = reinterpret_cast<float *>(s_sel + p.top);
		choose_experts(logits, p.correction, p.experts, p.top, s_choice, s_sel, s_val);
		zw = s_sel[z];
		if (blockIdx.x == 0 && part == 0 && z == 0) {
			for (int k = tid; k < p.top; k += NT) {
				float sum = 0.0f;
				for (int o = 0; o < p.top; o++) sum += s_val[o];
				p.sel[k] = s_sel[k];
				p.wgt[k] = s_val[k] / (sum + 1e-20f) * p.rscale;
			}
		}
	};
	if constexpr (PRO == TG_VP_EXPERT) choose(p.logits);

	const int group = KW == 4 ? (int)blockIdx.x : (int)blockIdx.x * 4 + w;  // tile group of this wave
	bool live = true;
	int tile0 = 0, tiles_here = 1;
	const Frag *W = nullptr;
	const Frag *R = nullptr;  // ROUTE: the router's matrix
	float late = 0.0f;        // a factor of the epilogue, requested with the weights (ROUTE: the lane's expert's correction)
	auto weights = [&] { W = reinterpret_cast<const Frag *>(p.W) + ((size_t)zw * p.zfrags + (size_t)tile0 * p.kfrags) * 64 + lane; };
	// the rest of the descriptor, in one batch, through the address of the argument block: made opaque here, so that no field can be
	// fetched earlier (which would end with a wait in front of the first loads)
	typedef const TgVec __attribute__((address_space(4))) *Desc;
	auto descriptor = [&] {
		Desc d = (Desc)((const char __attribute__((address_space(4))) *)__builtin_amdgcn_kernarg_segment_ptr() + VEC_DESC_OFFSET);
		asm volatile("" : "+s"(d) : : "memory");
		return d;
	};
	auto fetch_rest = [&] {
		const Desc d = descriptor();
		p.W = d->W;
		p.ntiles = d->ntiles;
		p.zfrags = d->zfrags;
		p.y = d->y;
		p.y_zstride = d->y_zstride;
		p.part_stride = d->part_stride;
		if constexpr (PRO == TG_VP_DYT || PRO == TG_VP_ROUTE || PRO == TG_VP_RMS) {
			p.mult = d->mult;
			p.x_out = d->x_out;
			p.h_out = d->h_out;
			if constexpr (PRO == TG_VP_RMS) p.width = d->width;
			else p.alpha = d->alpha;
		}
		if constexpr (PRO == TG_VP_RMS || PRO == TG_VP_HEADNORM) p.eps = d->eps;
		if constexpr (PRO == TG_VP_HEADNORM) {
			p.vdim = d->vdim;
			p.gate_sigmoid = d->gate_sigmoid;
		}
		if constexpr (PRO == TG_VP_ROUTE) {
			p.router = d->router;
			p.correction = d->correction;
			p.experts = d->experts;
			p.top = d->top;
		}
		if constexpr (EPI == TG_VE_LOGITS) {
			p.nout = d->nout;
			p.blk_val = d->blk_val;
			p.blk_idx = d->blk_idx;
		}
		if constexpr (EPI == TG_VE_GATE) p.gate = d->gate;
		if constexpr (EPI == TG_VE_WEIGHTED) p.wgt = d->wgt;
		if constexpr (EPI == TG_VE_STORE) p.bias = d->bias;
		live = group * NTL < p.ntiles;
		tile0 = live ? group * NTL : 0;
		tiles_here = min(NTL, p.ntiles - tile0);
		if constexpr (EPI == TG_VE_WEIGHTED) zw = p.sel[z];
		if constexpr (PRO != TG_VP_ROUTE) weights();
		if constexpr (PRO == TG_VP_ROUTE) R = reinterpret_cast<const Frag *>(p.router) + lane;
		if constexpr (EPI == TG_VE_GATE) late = p.gate[z];
		if constexpr (EPI == TG_VE_WEIGHTED) late = p.wgt[z];
	};
	const int step = KW, kf0 = kb + (KW == 4 ? w : 0);
	Frag wr[NTL][U];
	auto load = [&](int kf) {
#pragma unroll
		for (int u = 0; u < U; u++) {
			const int kk = kf + u * step, kc = min(kk, p.kfrags - 1);
#pragma unroll
			for (int t = 0; t < NTL; t++) {
				const Frag *at = W + ((size_t)(t < tiles_here ? t : 0) * p.kfrags + kc) * 64;
				// a head is read once per token: past the caches, which keep the layers' matrices
				wr[t][u] = KW == 1 ? __builtin_nontemporal_load(at) : *at;
			}
		}
	};

	// ROUTE: what is requested behind the inputs is the router's matrix (its rounds as in the product of its own that a router
	// of more tiles gets, so that the logits are the same); the experts' weights wait for the choice.
	constexpr int RU = PRO == TG_VP_ROUTE ? 8 : 1;
	Frag rt[RU];
	auto load_router = [&](int kf) {
#pragma unroll
		for (int u = 0; u < RU; u++) rt[u] = R[(size_t)min(kf + 4 * u, p.kfrags - 1) * 64];
	};
	auto load_first = [&] {
		fetch_rest();
		if constexpr (PRO == TG_VP_ROUTE) {
			load_router(w);
			late = p.correction[min(lane & 15, p.experts - 1)];  // (where it is used it was a round trip of its own, 0.4 us of 6.1)
		} else {
			load(kf0);
		}
	};

	// the vector's prologue: elements [k0, k0 + kn), then zeros that the surplus steps of the last round multiply
	if constexpr (PRO == TG_VP_PLAIN || PRO == TG_VP_EXPERT) {
		const float *x = p.x + (PRO == TG_VP_PLAIN ? (size_t)z * p.x_zstride : 0) + k0;
		for (int b = 0; b == 0 || b < kn; b += 8 * NT) {
			f32x4_t v[2];
#pragma unroll
			for (int i = 0; i < 2; i++) v[i] = tg_load4(x + min(b + 4 * (tid + i * NT), max(kn - 4, 0)));
			if (b == 0) load_first();
#pragma unroll
			for (int i = 0; i < 2; i++)
				if (b + 4 * (tid + i * NT) < kn) tg_store4(xs + b + 4 * (tid + i * NT), v[i]);
		}
	} else if constexpr (PRO == TG_VP_DYT || PRO == TG_VP_ROUTE) {
		int row = 0;
		if (p.embed) {
			const Desc d = descriptor();
			p.embed_ld = d->embed_ld;
			p.embed_scale = d->embed_scale;
			row = d->ctr[4];
			row = row < 0 ? 0 : (row >= d->vocab ? d->vocab - 1 : row);
		}
		// four elements per lane and pass; the padding behind the vector is zero in x, the parts, the norm and the table
		constexpr int PER = VP == 1 ? 1 : 2;
		{
			for (int b = 0; b == 0 || (VP == 3 && b < kn); b += 4 * PER * NT) {
				f32x4_t x[PER], nw[PER], nb[PER], add[PER];
				int c[PER];
#pragma unroll
				for (int i = 0; i < PER; i++) {
					c[i] = k0 + min(b + 4 * (tid + i * NT), max(kn - 4, 0));
					x[i] = p.embed ? tg_load4((const __bf16 *)p.embed + (size_t)row * p.embed_ld + c[i]) : tg_load4(p.x + c[i]);
					nw[i] = tg_load4(p.nw + c[i]);
					nb[i] = tg_load4(p.nb + c[i]);
					add[i] = f32x4_t{0, 0, 0, 0};
				}
				auto parts = [&](auto many, int q0) {
					constexpr int PQ = decltype(many)::value;
					f32x4_t pq[PER][PQ];
#pragma unroll
					for (int q = 0; q < PQ; q++)
#pragma unroll
						for (int i = 0; i < PER; i++) pq[i][q] = tg_load4(p.pend + (size_t)min(q0 + q, p.nparts - 1) * p.pend_stride + c[i]);
					if (b == 0 && q0 == 0) load_first();
#pragma unroll
					for (int q = 0; q < PQ; q++)
#pragma unroll
						for (int i = 0; i < PER; i++)
#pragma unroll
							for (int e = 0; e < 4; e++) add[i][e] += masked(pq[i][q][e], q0 + q < p.nparts);
				};
				if (p.nparts > 4) {
					for (int q0 = 0; q0 < p.nparts; q0 += 8) parts(Const<8>(), q0);
				} else if (p.nparts > 0) {
					parts(Const<4>(), 0);
				} else if (b == 0) {
					load_first();
				}
#pragma unroll
				for (int i = 0; i < PER; i++) {
					const int j = b + 4 * (tid + i * NT);
					f32x4_t h;
#pragma unroll
					for (int e = 0; e < 4; e++) {
						if (p.nparts) x[i][e] = x[i][e] + p.mult * add[i][e];
						h[e] = tanhf(p.alpha * x[i][e]) * nw[i][e] + nb[i][e];
					}
					if (j < kn) {
						tg_store4(xs + j, h);
						if (blockIdx.x == 0 && z == 0) {
							if (p.x_out) tg_store4(p.x_out + c[i], x[i]);
							if (p.h_out) tg_store4(p.h_out + c[i], h);
						}
					}
				}
			}
		}
	} else if constexpr (PRO == TG_VP_RMS) {
		// The whole vector in every workgroup (ksplit is 1): four elements per lane and pass; the first RP passes stay in
		// registers, the rest goes through LDS.  The padding is zero in x, the parts, the weights and the table.
		int row = 0;
		if (p.embed) {
			const Desc d = descriptor();
			p.embed_ld = d->embed_ld;
			p.embed_scale = d->embed_scale;
			row = d->ctr[4];
			row = row < 0 ? 0 : (row >= d->vocab ? d->vocab - 1 : row);
		}
		float *sv = reinterpret_cast<float *>(smem + sizeof(T) * (size_t)(per + KW * U) * TR::KF);  // [kn], wider vectors only
		const int npass = (kn + 4 * NT - 1) / (4 * NT);
		auto at = [&](int i) { return min(4 * (tid + i * NT), kn - 4); };
		auto source = [&](int c) {
			f32x4_t v;
			if (p.embed) {
				v = tg_load4((const __bf16 *)p.embed + (size_t)row * p.embed_ld + c);
#pragma unroll
				for (int e = 0; e < 4; e++) v[e] *= p.embed_scale;
			} else {
				v = tg_load4(p.x + c);
			}
			return v;
		};
		auto parts = [&](int c) {
			f32x4_t r = {0, 0, 0, 0};
			for (int q0 = 0; q0 < p.nparts; q0 += 8) {
				f32x4_t v[8];
#pragma unroll
				for (int q = 0; q < 8; q++) v[q] = tg_load4(p.pend + (size_t)min(q0 + q, p.nparts - 1) * p.pend_stride + c);
#pragma unroll
				for (int q = 0; q < 8; q++)
					if (q0 + q < p.nparts)
#pragma unroll
						for (int e = 0; e < 4; e++) r[e] += v[q][e];
			}
			return r;
		};
		auto total = [&](float v, int slot) {
			v = tg_wave_sum(v);
			if (lane == 0) s_misc[slot + w] = v;
			__syncthreads();
			return (s_misc[slot] + s_misc[slot + 1]) + (s_misc[slot + 2] + s_misc[slot + 3]);
		};
		constexpr int RP = VP == 1 ? 1 : 2;
		{
			f32x4_t x[RP], add[RP], nw[RP], pw[RP];
#pragma unroll
			for (int i = 0; i < RP; i++) {
				const int c = at(i);
				x[i] = source(c);
				nw[i] = tg_load4(p.nw + c);
				if (p.post) pw[i] = tg_load4(p.post + c);
			}
			auto first_parts = [&](auto many, int q0) {  // of all passes at once
				constexpr int PQ = decltype(many)::value;
				f32x4_t v[RP][PQ];
#pragma unroll
				for (int q = 0; q < PQ; q++)
#pragma unroll
					for (int i = 0; i < RP; i++) v[i][q] = tg_load4(p.pend + (size_t)min(q0 + q, p.nparts - 1) * p.pend_stride + at(i));
				if (VP == 1 && q0 == 0) load_first();
#pragma unroll
				for (int q = 0; q < PQ; q++)
#pragma unroll
					for (int i = 0; i < RP; i++)
#pragma unroll
						for (int e = 0; e < 4; e++) add[i][e] += masked(v[i][q][e], q0 + q < p.nparts);
			};
#pragma unroll
			for (int i = 0; i < RP; i++) add[i] = f32x4_t{0, 0, 0, 0};
			// A vector of one pass has its weights requested next to it, a longer one when it is there (1152 columns, 648
			// workgroups: 9.05 us against 9.45; width 640 in fp32: 5.5 against 5.8)
			if (p.nparts > 4) {
				for (int q0 = 0; q0 < p.nparts; q0 += 8) first_parts(Const<8>(), q0);
			} else if (p.nparts > 0) {
				first_parts(Const<4>(), 0);
			} else if (VP == 1) {
				load_first();
			}
			if constexpr (VP != 1) load_first();
			if (!p.post) {
#pragma unroll
				for (int i = 0; i < RP; i++) pw[i] = f32x4_t{p.mult, p.mult, p.mult, p.mult};
			}
			auto wide = [&](int i, auto &&f) {  // f(column, its four values in LDS)
				if constexpr (VP == 3)
					for (; i < npass; i++) {
						const int j = 4 * (tid + i * NT);
						if (j < kn) f(j);
					}
			};
			if (p.nparts) {
				float inv = 1.0f;
				if (p.post) {
					float ss = 0.0f;
#pragma unroll
					for (int i = 0; i < RP; i++)
						if (4 * (tid + i * NT) < kn)
#pragma unroll
							for (int e = 0; e < 4; e++) ss = fmaf(add[i][e], add[i][e], ss);
					wide(RP, [&](int j) {
						const f32x4_t v = parts(j);
#pragma unroll
						for (int e = 0; e < 4; e++) ss = fmaf(v[e], v[e], ss);
						tg_store4(sv + j, v);
					});
					inv = 1.0f / sqrtf(total(ss, 0) / (float)p.width + p.eps);
				} else {
					wide(RP, [&](int j) { tg_store4(sv + j, parts(j)); });
				}
#pragma unroll
				for (int i = 0; i < RP; i++)
#pragma unroll
					for (int e = 0; e < 4; e++) x[i][e] += add[i][e] * inv * pw[i][e];
				wide(RP, [&](int j) {
					f32x4_t v = source(j);
					const f32x4_t a = tg_load4(sv + j), b = p.post ? tg_load4(p.post + j) : f32x4_t{p.mult, p.mult, p.mult, p.mult};
#pragma unroll
					for (int e = 0; e < 4; e++) v[e] += a[e] * inv * b[e];
					tg_store4(sv + j, v);
				});
			} else {
				wide(RP, [&](int j) { tg_store4(sv + j, source(j)); });
			}
			float ss = 0.0f;
#pragma unroll
			for (int i = 0; i < RP; i++)
				if (4 * (tid + i * NT) < kn)
#pragma unroll
					for (int e = 0; e < 4; e++) ss = fmaf(x[i][e], x[i][e], ss);
			wide(RP, [&](int j) {
				const f32x4_t v = tg_load4(sv + j);
#pragma unroll
				for (int e = 0; e < 4; e++) ss = fmaf(v[e], v[e], ss);
			});
			const float inv = 1.0f / sqrtf(total(ss, 4) / (float)p.width + p.eps);
			const bool first = blockIdx.x == 0 && z == 0;
			auto finish = [&](int j, f32x4_t v, f32x4_t n) {
				f32x4_t h;
#pragma unroll
				for (int e = 0; e < 4; e++) h[e] = v[e] * inv * n[e];
				tg_store4(xs + j, h);
				if (first && p.x_out) tg_store4(p.x_out + j, v);
				if (first && p.h_out) tg_store4(p.h_out + j, h);
			};
#pragma unroll
			for (int i = 0; i < RP; i++)
				if (4 * (tid + i * NT) < kn) finish(4 * (tid + i * NT), x[i], nw[i]);
			wide(RP, [&](int j) { finish(j, tg_load4(sv + j), tg_load4(p.nw + j)); });
		}
	} else if constexpr (PRO == TG_VP_HEADNORM) {
		// head by head, a wave each, four elements per lane and pass: sum of squares, then the head's elements that lie in
		// this part of K
		const int h_lo = k0 / p.vdimp, h_hi = min((k0 + kn - 1) / p.vdimp, p.heads16 - 1), vl = p.vdimp - 4;
		bool first = true;
		for (int a = h_lo + w; a <= h_hi; a += 4) {
			const float *o = p.x + (size_t)a * p.vdimp, *g = p.gate + (size_t)a * p.vdimp;
			const f32x4_t o0 = tg_load4(o + min(4 * lane, vl)), g0 = tg_load4(g + min(4 * lane, vl)), w0 = tg_load4(p.nw + min(4 * lane, vl));
			if (first) load_first();
			first = false;
			float ss = 0.0f;
			for (int v = 4 * lane; v < p.vdimp; v += 256) {  // the padding is zero
				const f32x4_t ov = v < 256 ? o0 : tg_load4(o + v);
#pragma unroll
				for (int e = 0; e < 4; e++) ss = fmaf(ov[e], ov[e], ss);
			}
			ss = tg_wave_sum(ss);
			const float inv = 1.0f / sqrtf(ss / (float)p.vdim + p.eps);
			for (int v = 4 * lane; v < p.vdimp; v += 256) {
				const f32x4_t ov = v < 256 ? o0 : tg_load4(o + v), gv = v < 256 ? g0 : tg_load4(g + v), wv = v < 256 ? w0 : tg_load4(p.nw + v);
				const int j = a * p.vdimp + v - k0;
				f32x4_t r;
#pragma unroll
				for (int e = 0; e < 4; e++) r[e] = ov[e] * inv * wv[e] * (p.gate_sigmoid ? tg_sigmoid(gv[e]) : tg_silu(gv[e]));
				if (j >= 0 && j < kn) tg_store4(xs + j, r);
			}
		}
		if (first) load_first();
		for (int j = tid; j < kn; j += NT)
			if ((k0 + j) / p.vdimp >= p.heads16) xs[j] = (T)0.0f;
	} else if constexpr (PRO == TG_VP_MERGE_HEADS) {
		// a row of 16 lanes per head: the factors of its partials; then element by element
		__shared__ float s_f[TG_VEC_MERGE_HEADS_MAX][TG_VEC_MERGE_MAX];
		const int g16 = (p.group + 15) / 16 * 16, bl = min(lane & 15, p.nmerge - 1);
		auto padded = [&](int h) { const int g = h / p.group; return g * g16 + h - g * p.group; };
		const int h_lo = min(k0 / p.vdimp, p.heads - 1), h_hi = min((k0 + max(kn, 1) - 1) / p.vdimp, p.heads - 1);
		auto column = [&](int j) {
			const int k = k0 + j, h = min(k / p.vdimp, p.heads - 1);
			return p.part_acc + (size_t)padded(h) * p.x_zstride + min(k - h * p.vdimp, p.vdimp - 1);
		};
		const size_t step_b = (size_t)p.heads16 * p.x_zstride;
		const int ha = min(h_lo + 4 * w + (lane >> 4), h_hi);
		float2 ml = *reinterpret_cast<const float2 *>(p.part_ml + ((size_t)bl * p.heads16 + padded(ha)) * 2);
		float a[TG_VEC_MERGE_MAX];
		const float *pa = column(min(tid, max(kn - 1, 0)));
#pragma unroll
		for (int b = 0; b < TG_VEC_MERGE_MAX; b++) a[b] = pa[(size_t)min(b, p.nmerge - 1) * step_b];
		load_first();
		const bool in = (lane & 15) < p.nmerge;
		for (int hb = h_lo; hb <= h_hi; hb += 16) {
			const int h = min(hb + 4 * w + (lane >> 4), h_hi);
			if (hb != h_lo) ml = *reinterpret_cast<const float2 *>(p.part_ml + ((size_t)bl * p.heads16 + padded(h)) * 2);
			const float m = tg_row16_max(in ? ml.x : -INFINITY);
			const float f = in ? expf(ml.x - m) : 0.0f;
			const float inv = 1.0f / tg_row16_sum(f * ml.y);
			s_f[h - h_lo][lane & 15] = f * inv;
		}
		__syncthreads();
		for (int j = tid; j < kn; j += NT) {
			const int h = (k0 + j) / p.vdimp;
			if (j != tid) {
				pa = column(j);
#pragma unroll
				for (int b = 0; b < TG_VEC_MERGE_MAX; b++) a[b] = pa[(size_t)min(b, p.nmerge - 1) * step_b];
			}
			float r = 0.0f;
			if (h < p.heads)
#pragma unroll
				for (int b = 0; b < TG_VEC_MERGE_MAX; b++) r = fmaf(s_f[h - h_lo][b], a[b], r);
			xs[j] = (T)r;
		}
	} else {  // MERGE: at most 16 partials
		const int bl = min(lane & 15, p.nmerge - 1);
		const float2 ml = *reinterpret_cast<const float2 *>(p.part_ml + ((size_t)bl * p.heads16 + z) * 2);
		float a[TG_VEC_MERGE_MAX];
		const float *pa = p.part_acc + (size_t)z * p.x_zstride + k0;
#pragma unroll
		for (int b = 0; b < TG_VEC_MERGE_MAX; b++)
			a[b] = pa[(size_t)min(b, p.nmerge - 1) * p.heads16 * p.x_zstride + min(tid, max(kn - 1, 0))];
		load_first();
		const bool in = (lane & 15) < p.nmerge;
		const float m = tg_row16_max(in ? ml.x : -INFINITY);
		const float f = in ? expf(ml.x - m) : 0.0f;
		const float inv = 1.0f / tg_row16_sum(f * ml.y);
		if (tid < 16) s_misc[tid] = f * inv;
		__syncthreads();
		for (int j = tid; j < kn; j += NT) {
			float r = 0.0f;
#pragma unroll
			for (int b = 0; b < TG_VEC_MERGE_MAX; b++) {
				if (j != tid) a[b] = pa[(size_t)min(b, p.nmerge - 1) * p.heads16 * p.x_zstride + j];
				r = fmaf(s_misc[b], a[b], r);
			}
			xs[j] = (T)r;
		}
	}
	for (int j = kn + tid; j < kn + KW * U * TR::KF; j += NT) xs[j] = (T)0.0f;
	__syncthreads();
	if constexpr (PRO == TG_VP_ROUTE) {
		f32x4_t ra = {0, 0, 0, 0};
		for (int kf = w; kf < p.kfrags; kf += 4 * RU) {
			if (kf != w) load_router(kf);
#pragma unroll
			for (int u = 0; u < RU; u++) {
				if (kf + 4 * u >= p.kfrags) break;
				const Frag xf = *reinterpret_cast<const Frag *>(xs + (size_t)(kf + 4 * u) * TR::KF + (lane >> 4) * TR::KV);
				ra = TR::mma(xf, rt[u], ra);
			}
		}
		if (lane < 16) s_misc[16 * w + lane] = ra[0];  // (not s_red: a wave without weights of its own may be in the epilogue while another reads these)
		__syncthreads();
		// the choice of choose_experts for at most 16 experts, expert = lane, by every wave for itself: nothing goes through LDS
		const int e = lane & 15;
		const float logit = (s_misc[e] + s_misc[16 + e]) + (s_misc[32 + e] + s_misc[48 + e]);
		const bool is = e < p.experts;
		const float val = tg_sigmoid(logit), score = is ? tg_choice_score(val, late) : -INFINITY;
		int rank = 0;
#pragma unroll
		for (int o = 0; o < 16; o++) {
			const float other = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(score), o));
			rank += (other > score || (other == score && o < e)) ? 1 : 0;
		}
		auto chosen = [&](int k) {  // the lane of the k-th choice (every rank of 0 .. 15 is there once, the padding's behind the experts')
			return __builtin_ctzll(__ballot(rank == k));
		};
		zw = chosen(z);
		if (blockIdx.x == 0 && part == 0 && z == 0 && w == 0) {
			float sum = 0.0f;
			for (int k = 0; k < p.top; k++) sum += __shfl(val, chosen(k), 64);
			if (lane < 16 && rank < p.top) {
				p.sel[rank] = e;
				p.wgt[rank] = val / (sum + 1e-20f) * p.rscale;
			}
		}
		weights();
		load(kf0);
	}

	f32x4_t acc[NTL];
#pragma unroll
	for (int t = 0; t < NTL; t++) acc[t] = f32x4_t{0, 0, 0, 0};
	const T *xl = xs + (lane >> 4) * TR::KV;
	for (int kf = kf0; kf < ke; kf += step * U) {
		Frag cur[NTL][U];
#pragma unroll
		for (int t = 0; t < NTL; t++)
#pragma unroll
			for (int u = 0; u < U; u++) cur[t][u] = wr[t][u];
		if (kf + step * U < ke) load(kf + step * U);
#pragma unroll
		for (int u = 0; u < U; u++) {
			const Frag xf = *reinterpret_cast<const Frag *>(xl + (size_t)(kf + u * step - kb) * TR::KF);
#pragma unroll
			for (int t = 0; t < NTL; t++) acc[t] = TR::mma(xf, cur[t][u], acc[t]);
		}
	}
	// all 16 rows of the first operand are the vector: element 0 of lane l is output l % 16 of the tile
	if constexpr (KW == 4) {
		if (lane < 16) {
#pragma unroll
			for (int t = 0; t < NTL; t++) s_red[w][t * 16 + lane] = acc[t][0];
		}
		__syncthreads();
		if (tid < 16) {
			float v[NTL];
#pragma unroll
			for (int t = 0; t < NTL; t++) v[t] = (s_red[0][t * 16 + tid] + s_red[1][t * 16 + tid]) + (s_red[2][t * 16 + tid] + s_red[3][t * 16 + tid]);
			float *y = p.y + (size_t)part * p.part_stride + (size_t)z * p.y_zstride;
			if constexpr (EPI == TG_VE_SWIGLU) {
				y[group * 16 + tid] = tg_silu(v[0]) * v[NTL - 1];
			} else {
				float r = v[0];
				if constexpr (EPI == TG_VE_STORE) {
					if (p.bias) {
						r += p.bias[group * NTL * 16 + tid];
						if constexpr (NTL == 2) {
							if (group * 2 + 1 < p.ntiles) v[1] += p.bias[group * 32 + 16 + tid];
						}
					}
				}
				if constexpr (EPI == TG_VE_GELU) r = tg_gelu(r);
				if constexpr (EPI == TG_VE_GATE) r *= tg_sigmoid(late);
				if constexpr (EPI == TG_VE_WEIGHTED) r *= late;
				y[group * NTL * 16 + tid] = r;
				if constexpr (NTL == 2) {
					if (group * 2 + 1 < p.ntiles) y[group * 32 + 16 + tid] = v[1];
				}
				if constexpr (EPI == TG_VE_LOGITS) {
					float bv = group * 16 + tid < p.nout ? r : -INFINITY;
					int bi = group * 16 + tid;
#pragma unroll
					for (int o = 8; o > 0; o >>= 1) {
						const float ov = __shfl_xor(bv, o, 16);
						const int oi = __shfl_xor(bi, o, 16);
						if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
					}
					if (tid == 0) { p.blk_val[blockIdx.x] = bv; p.blk_idx[blockIdx.x] = bi; }
				}
			}
		}
	} else {
		if (lane < 16) {
			const int o = group * 16 + lane;
			float r = acc[0][0];
			if constexpr (EPI == TG_VE_STORE) {
				if (p.bias && live) r += p.bias[o];
			}
			if (live) p.y[(size_t)z * p.y_zstride + o] = r;
			if constexpr (EPI == TG_VE_LOGITS) s_red[w][lane] = live && o < p.nout ? r : -INFINITY;
		}
		if constexpr (EPI == TG_VE_LOGITS) {
			__syncthreads();
			if (tid < 64) {
				float bv = s_red[tid >> 4][tid & 15];
				int bi = (int)blockIdx.x * 64 + tid;
#pragma unroll
				for (int o = 32; o > 0; o >>= 1) {
					const float ov = __shfl_xor(bv, o, 64);
					const int oi = __shfl_xor(bi, o, 64);
					if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
				}
				if (tid == 0) { p.blk_val[blockIdx.x] = bv; p.blk_idx[blockIdx.x] = bi; }
			}
		}
	}
}

bool vec_wide(const TgVec &v, int epi) { return (epi == TG_VE_STORE || epi == TG_VE_LOGITS) && v.ksplit == 1 && v.nz == 1 && v.ntiles >= 2048; }

// Two tiles per workgroup where one each would be two workgroups per compute unit and more: the prologue (with its reads of
// the parts of the residual) is done half as often.
bool vec_pairs(const TgVec &v, int epi) { return epi == TG_VE_STORE && v.nparts > 0 && v.nz == 1 && v.ksplit == 1 && v.ntiles >= 448; }

// the norm's vector beyond what the registers of a workgroup hold
size_t rms_lds(int pro, int k) { return pro == TG_VP_RMS && k > 8 * NT ? sizeof(float) * (size_t)k : 0; }

// How many passes of 1024 elements a norm's prologue takes: 1, 2, or more (3).  A prologue requests the inputs of all its passes
// before it uses one, also for lanes behind the vector's end: with two passes of eight parts each for every vector, the 4096
// workgroups of a head of width 640 read as many bytes for their norms as for the weights (72 us; 66 with what there is).  The
// classes are instances and not branches because a launch pays for the instructions it fetches: with both in one kernel the
// 5.2 us products of width 1152 took 6.4.
int vec_class(int pro, int k) { return pro != TG_VP_DYT && pro != TG_VP_RMS && pro != TG_VP_ROUTE ? 0 : k <= 4 * NT ? 1 : k <= 8 * NT ? 2 : 3; }

// Fragments in flight for n of them a wave: all where they fit, else as few equal rounds as possible; whether some n of a range
// gets u (instances that no length of a class reaches are not built: a third of the library's size).
constexpr int vec_depth(int n) {
	return n <= 2 ? 2 : n <= 4 ? 4 : n <= 6 || (n > 9 && n <= 12) ? 6 : n <= 8 || (n > 12 && n <= 16) || (n > 18 && n <= 24) ? 8 : 9;
}
constexpr bool vec_reaches(int u, int n_min, int n_max) {
	for (int n = n_min; n <= n_max && n <= n_min + 32; n++)
		if (vec_depth(n) == u) return true;
	return false;
}

template <class TR, int PRO, int EPI, int VP>
void launch_vec_vp(const TgVec &v, hipStream_t s) {
	// fragments a wave in this class
	constexpr int PASS = 4 * NT / TR::KF / 4, ROUTED = (TG_ROUTE_ROW_MAX / (int)sizeof(typename TR::T) / TR::KF + 3) / 4;
	constexpr int N_MIN = VP == 3 ? 2 * PASS + 1 : VP == 2 ? PASS + 1 : 1, N_CLASS = VP == 1 ? PASS : VP == 2 ? 2 * PASS : 1 << 16;
	constexpr int N_MAX = PRO == TG_VP_ROUTE && ROUTED < N_CLASS ? ROUTED : N_CLASS;
	const VecHot h = vec_hot<PRO, EPI>(v);
#define TG_VEC_LAUNCH(ntl, kw, u, grid, pad)                                                                                                       \
	hipLaunchKernelGGL((vec_kernel<TR, PRO, EPI, ntl, kw, u, VP>), grid, dim3(NT), lds(pad), s, h.a[0], h.a[1], h.a[2], h.a[3], h.i[0], h.i[1], \
	                   h.i[2], h.i[3], h.i[4], h.i[5], v)
	constexpr int NTL = EPI == TG_VE_SWIGLU ? 2 : 1;
	const int per = (v.kfrags + v.ksplit - 1) / v.ksplit;
	if constexpr ((PRO == TG_VP_DYT || PRO == TG_VP_RMS) && EPI == TG_VE_STORE) {
		if (!vec_wide(v, EPI) && vec_pairs(v, EPI)) {
			const int n = (per + 3) / 4;
			auto lds = [&](int pad) { return sizeof(typename TR::T) * (size_t)(per + pad) * TR::KF + rms_lds(PRO, per * TR::KF); };
			const dim3 grid((unsigned)tg_vec_blocks(v, EPI), (unsigned)v.ksplit, (unsigned)v.nz);
			if constexpr (N_MIN <= 6) {
				if (n <= 6) {
					TG_VEC_LAUNCH(2, 4, 6, (grid), 24);
					return;
				}
			}
			TG_VEC_LAUNCH(2, 4, 8, (grid), 32);
			return;
		}
	}
	const unsigned bx = (unsigned)tg_vec_blocks(v, EPI);
	auto lds = [&](int pad) {
		size_t b = sizeof(typename TR::T) * (size_t)(per + pad) * TR::KF;
		b += rms_lds(PRO, per * TR::KF);
		if (PRO == TG_VP_EXPERT) b += sizeof(float) * (size_t)(((v.experts + 3) & ~3) + 2 * v.top);
		return b;
	};
	if constexpr (EPI == TG_VE_STORE || EPI == TG_VE_LOGITS) {
		if (vec_wide(v, EPI)) {
			TG_VEC_LAUNCH(1, 1, 8, (dim3(bx, 1, 1)), 8);
			return;
		}
	}
	const dim3 grid(bx, (unsigned)v.ksplit, (unsigned)v.nz);
	const int depth = vec_depth((per + 3) / 4);
	auto go = [&](auto u) {
		constexpr int U = decltype(u)::value;
		if constexpr (vec_reaches(U, N_MIN, N_MAX)) {
			if (depth == U) TG_VEC_LAUNCH(NTL, 4, U, (grid), 4 * U);
		}
	};
	go(Const<2>());
	go(Const<4>());
	go(Const<6>());
	go(Const<8>());
	go(Const<9>());
}

#undef TG_VEC_LAUNCH

template <class TR, int PRO, int EPI>
void launch_vec_t(const TgVec &v, hipStream_t s) {
	if constexpr (PRO == TG_VP_DYT || PRO == TG_VP_RMS || PRO == TG_VP_ROUTE) {
		const int c = vec_class(PRO, (v.kfrags + v.ksplit - 1) / v.ksplit * TR::KF);
		if (c == 1) launch_vec_vp<TR, PRO, EPI, 1>(v, s);
		else if (c == 2) launch_vec_vp<TR, PRO, EPI, 2>(v, s);
		else launch_vec_vp<TR, PRO, EPI, 3>(v, s);
	} else {
		launch_vec_vp<TR, PRO, EPI, 0>(v, s);
	}
}

template <class TR>
void launch_vec_dt(const TgVec &v, int pro, int epi, hipStream_t s) {
	if (pro == TG_VP_PLAIN && epi == TG_VE_STORE) launch_vec_t<TR, TG_VP_PLAIN, TG_VE_STORE>(v, s);
	else if (pro == TG_VP_DYT && epi == TG_VE_STORE) launch_vec_t<TR, TG_VP_DYT, TG_VE_STORE>(v, s);
	else if (pro == TG_VP_DYT && epi == TG_VE_LOGITS) launch_vec_t<TR, TG_VP_DYT, TG_VE_LOGITS>(v, s);
	else if (pro == TG_VP_RMS && epi == TG_VE_STORE) launch_vec_t<TR, TG_VP_RMS, TG_VE_STORE>(v, s);
	else if (pro == TG_VP_RMS && epi == TG_VE_GELU) launch_vec_t<TR, TG_VP_RMS, TG_VE_GELU>(v, s);
	else if (pro == TG_VP_RMS && epi == TG_VE_LOGITS) launch_vec_t<TR, TG_VP_RMS, TG_VE_LOGITS>(v, s);
	else if (pro == TG_VP_MERGE && epi == TG_VE_STORE) launch_vec_t<TR, TG_VP_MERGE, TG_VE_STORE>(v, s);
	else if (pro == TG_VP_MERGE_HEADS) launch_vec_t<TR, TG_VP_MERGE_HEADS, TG_VE_STORE>(v, s);
	else if (pro == TG_VP_HEADNORM) launch_vec_t<TR, TG_VP_HEADNORM, TG_VE_STORE>(v, s);
	else if (pro == TG_VP_MERGE) launch_vec_t<TR, TG_VP_MERGE, TG_VE_GATE>(v, s);
	else if (pro == TG_VP_EXPERT) launch_vec_t<TR, TG_VP_EXPERT, TG_VE_SWIGLU>(v, s);
	else if (pro == TG_VP_ROUTE) launch_vec_t<TR, TG_VP_ROUTE, TG_VE_SWIGLU>(v, s);
	else if (pro == TG_VP_PLAIN && epi == TG_VE_GATE) launch_vec_t<TR, TG_VP_PLAIN, TG_VE_GATE>(v, s);
	else launch_vec_t<TR, TG_VP_PLAIN, TG_VE_WEIGHTED>(v, s);
}

// ---- tiled products --------------------------------------------------------------------------------------------------------
// A workgroup computes BM x BN with WM x WN waves of (16 MI) x (16 NI) each.  K advances by two fragments (128 bytes of a
// row) per stage: both operands go global -> registers -> LDS in fragment order (two LDS buffers, two sets of registers: the
// loads of the next two stages are in flight during the matrix instructions of this one), one LDS-only barrier per stage.
template <class TR, int EPI, int WM, int WN, int MI, int NI, bool GROUPED>
__global__ __launch_bounds__(256, 2) void linear_kernel(TgGemm g) {
	typedef typename TR::T T;
	typedef typename TR::Frag Frag;
	constexpr int BM = WM * MI * 16, BN = WN * NI * 16;
	constexpr int AF = BM / 16, BF = BN / 16, NF = 2 * (AF + BF), PW = NF / 4;  // fragments per stage, per wave
	static_assert(NF % 4 == 0 && WM * WN == 4, "four waves share a stage's fragments");
	__shared__ __align__(16) Frag lds[2][NF * 64];
	const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int ntn = (g.N + BN - 1) / BN;
	constexpr bool PARTS = EPI == TG_GE_F32 && !GROUPED && BM == 32;

	// Workgroups go to the 8 XCDs in turn: give each XCD a contiguous run of the tile order, so that the workgroups it
	// runs side by side share weight tiles and activation rows in its L2.  (A list of groups launches as many workgroups
	// as it could have tiles: the run lengths come from the tiles it has.)
	const int mrows = EPI == TG_GE_TRANS ? g.rows_out : g.M;
	const int ntm = GROUPED ? *g.ntiles : (mrows + BM - 1) / BM;
	int b;
	{
		const int total = ntm * ntn * (PARTS ? g.kparts : 1), q = total >> 3, r = total & 7, x = (int)blockIdx.x & 7, i = (int)blockIdx.x >> 3;
		if (i >= q + (x < r ? 1 : 0)) return;
		b = x * q + min(x, r) + i;
	}
	int m0, m1, tn, part = 0;
	const Frag *W = reinterpret_cast<const Frag *>(g.W);
	if constexpr (PARTS) {
		part = b / (ntm * ntn);
		b -= part * ntm * ntn;
	}
	if constexpr (GROUPED) {
		const int t = b / ntn;
		tn = b - t * ntn;
		const int4 tile = g.tiles[t];
		m0 = tile.y;
		m1 = tile.z;
		W += (size_t)tile.x * g.group_frags * 64;
	} else {
		tn = b / ntm;
		m0 = (b - tn * ntm) * BM;
		m1 = g.M;
	}
	const int kfr = g.K / TR::KF, nfr = g.N / 16;
	int nst = kfr / 2, s0 = 0;  // stages of this workgroup, the first of them
	if constexpr (PARTS) {
		const int per = (nst + g.kparts - 1) / g.kparts;
		s0 = part * per;
		nst = min(per, nst - s0);  // (tg_linear_kparts leaves no part empty)
	}

	// this wave's fragments of a stage: f = w * PW + i; the first 2 AF are A (row tile f / 2, k half f % 2), then B
	// (addresses: a base that the wave shares, 32-bit offsets per lane; operands are below 4 GiB)
	const unsigned char *base[PW];
	unsigned off[PW];
	int adv[PW];
#pragma unroll
	for (int i = 0; i < PW; i++) {
		const int f = w * PW + i;
		if (f < 2 * AF) {
			int r = min(m0 + (f >> 1) * 16 + (lane & 15), m1 - 1);
			if (g.row_src) r = g.row_src[r];
			base[i] = reinterpret_cast<const unsigned char *>(g.A) + (f & 1) * 64;
			off[i] = (unsigned)r * (unsigned)(g.lda * (int)sizeof(T)) + (unsigned)(lane >> 4) * 16u;
			adv[i] = 128;
		} else {
			const int fb = f - 2 * AF, nf = min(tn * BF + (fb >> 1), nfr - 1);
			base[i] = reinterpret_cast<const unsigned char *>(W + ((size_t)nf * kfr + (fb & 1)) * 64);
			off[i] = (unsigned)lane * 16u;
			adv[i] = 2048;
		}
		if constexpr (PARTS) base[i] += (size_t)s0 * adv[i];
	}
	Frag st[2][PW];
	auto fetch = [&](int set, int s) {
		s = min(s, nst - 1);
#pragma unroll
		for (int i = 0; i < PW; i++) st[set][i] = *reinterpret_cast<const Frag *>(base[i] + (size_t)s * adv[i] + off[i]);
	};
	auto put = [&](int set) {
#pragma unroll
		for (int i = 0; i < PW; i++) lds[set][(w * PW + i) * 64 + lane] = st[set][i];
	};
	const int wm = w / WN, wn = w - wm * WN;
	f32x4_t acc[MI][NI];
#pragma unroll
	for (int i = 0; i < MI; i++)
#pragma unroll
		for (int j = 0; j < NI; j++) acc[i][j] = f32x4_t{0, 0, 0, 0};

	// Two sets of operand registers as well: the LDS reads of one half of a stage are in flight during the matrix
	// instructions of the half before it.
	Frag fa[2][MI], fb[2][NI];
	auto read = [&](int kh, int par) {
#pragma unroll
		for (int i = 0; i < MI; i++) fa[kh][i] = lds[par][((wm * MI + i) * 2 + kh) * 64 + lane];
#pragma unroll
		for (int j = 0; j < NI; j++) fb[kh][j] = lds[par][(2 * AF + (wn * NI + j) * 2 + kh) * 64 + lane];
	};
	auto multiply = [&](int kh) {
#pragma unroll
		for (int i = 0; i < MI; i++)
#pragma unroll
			for (int j = 0; j < NI; j++)
				acc[i][j] = EPI == TG_GE_TRANS ? TR::mma(fa[kh][i], fb[kh][j], acc[i][j]) : TR::mma(fb[kh][j], fa[kh][i], acc[i][j]);
	};
	fetch(0, 0);
	fetch(1, 1);
	put(0);
	fetch(0, 2);
	tg_lds_barrier();
	read(0, 0);
	// LDS buffer and register set of a stage: its parity
	// (the order is pinned: left to itself the scheduler moves every LDS read down to its use)
	constexpr int MM = MI * NI * (TR::DT == TG_DT_BF16 ? 1 : 4), RD = MI + NI;
	constexpr int MR = MM / 2 / RD > 0 ? MM / 2 / RD : 1, MP = MM / 2 / PW > 0 ? MM / 2 / PW : 1;
	auto stage = [&](int s, int par) {
		read(1, par);
		multiply(0);
		put(par ^ 1);
		fetch(par ^ 1, s + 3);
#pragma unroll
		for (int i = 0; i < RD; i++) {
			__builtin_amdgcn_sched_group_barrier(0x100, 1, 0);        // LDS read
			__builtin_amdgcn_sched_group_barrier(0x008, MR, 0);  // matrix instructions
		}
#pragma unroll
		for (int i = 0; i < PW; i++) {
			__builtin_amdgcn_sched_group_barrier(0x008, MP, 0);
			__builtin_amdgcn_sched_group_barrier(0x200, 1, 0);        // LDS write
			__builtin_amdgcn_sched_group_barrier(0x020, 1, 0);        // global load
		}
		__builtin_amdgcn_sched_barrier(0);
		tg_lds_barrier();
		__builtin_amdgcn_sched_barrier(0);
		read(0, par ^ 1);
		multiply(1);
#pragma unroll
		for (int i = 0; i < RD; i++) {
			__builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
			__builtin_amdgcn_sched_group_barrier(0x008, MM / RD > 0 ? MM / RD : 1, 1);
		}
		__builtin_amdgcn_sched_barrier(0);
	};
	// (pairs without a branch between them: across one, the waits for the older register set would cover the newer one too)
	int s = 0;
	for (; s + 1 < nst; s += 2) {
		stage(s, 0);
		stage(s + 1, 1);
	}
	if (s < nst) stage(s, 0);

	const int lr = lane & 15, lg = lane >> 4;
	if constexpr (EPI == TG_GE_TRANS) {
		// lane: column n = lr, rows m = 4 lg + i, four consecutive keys of a 32-key (bf16) or 16-key (fp32) operand block
#pragma unroll
		for (int i = 0; i < MI; i++)
#pragma unroll
			for (int j = 0; j < NI; j++) {
				const int n = tn * BN + (wn * NI + j) * 16 + lr, m = m0 + (wm * MI + i) * 16 + 4 * lg;
				if (n >= g.N || m >= g.rows_out) continue;
				int at = m;
				if constexpr (TR::DT == TG_DT_BF16) at = (m & ~31) + lg * 8 + ((m >> 4) & 1) * 4;
				tg_store4((T *)g.C + (size_t)n * g.ldc + at, acc[i][j]);
			}
	} else {
		// lane: row m = lr, columns n = 4 lg + i
#pragma unroll
		for (int i = 0; i < MI; i++) {
			const int m = m0 + (wm * MI + i) * 16 + lr;
			if (m >= m1) continue;
			if constexpr (EPI == TG_GE_SWIGLU) {
#pragma unroll
				for (int j = 0; j < NI; j += 2) {
					const int n = tn * BN + (wn * NI + j) * 16;  // of the interleaved rows
					if (n >= g.N) continue;
					f32x4_t r;
#pragma unroll
					for (int e = 0; e < 4; e++) r[e] = tg_silu(acc[i][j][e]) * acc[i][j + 1][e];
					tg_store4((T *)g.C + (size_t)m * g.ldc + n / 2 + 4 * lg, r);
				}
			} else {
#pragma unroll
				for (int j = 0; j < NI; j++) {
					const int n = tn * BN + (wn * NI + j) * 16 + 4 * lg;
					if (n >= g.N) continue;
					if constexpr (EPI == TG_GE_STORE) {
						if (g.bias && n < g.n_split) {
							const f32x4_t b = tg_load4(g.bias + n);
#pragma unroll
							for (int e = 0; e < 4; e++) acc[i][j][e] += b[e];
						}
						if (n < g.n_split) tg_store4((T *)g.C + (size_t)m * g.ldc + n, acc[i][j]);
						else tg_store4(g.C2 + (size_t)m * g.ldc2 + n - g.n_split, acc[i][j]);
					} else if constexpr (EPI == TG_GE_GELU) {
						f32x4_t r;
#pragma unroll
						for (int e = 0; e < 4; e++) r[e] = tg_gelu(acc[i][j][e]);
						tg_store4((T *)g.C + (size_t)m * g.ldc + n, r);
					} else if constexpr (EPI == TG_GE_F32) {
						tg_store4(g.C2 + (PARTS ? (size_t)part * g.part_stride : 0) + (size_t)m * g.ldc2 + n, acc[i][j]);
					} else {
						float *c = g.C2 + (size_t)m * g.ldc2 + n;
						f32x4_t x = tg_load4(c);
#pragma unroll
						for (int e = 0; e < 4; e++) x[e] = x[e] + g.mult * acc[i][j][e];
						tg_store4(c, x);
					}
				}
			}
		}
	}
}

// Few columns (a router): 16 rows x 64 columns per workgroup, the waves share K, operands straight from memory in fragment
// order, partial sums meet in LDS.
template <class TR>
__global__ __launch_bounds__(256) void linear_thin_kernel(TgGemm g) {
	typedef typename TR::T T;
	typedef typename TR::Frag Frag;
	constexpr int NI = 4, U = 4;
	__shared__ f32x4_t s_acc[4][NI][64];
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, lg = lane >> 4;
	const int m0 = blockIdx.x * 16, n0 = blockIdx.y * NI, kfr = g.K / TR::KF, nfr = g.N / 16;
	const T *A = (const T *)g.A + (size_t)min(m0 + lr, g.M - 1) * g.lda + lg * TR::KV;
	const Frag *W = reinterpret_cast<const Frag *>(g.W) + lane;
	f32x4_t acc[NI];
#pragma unroll
	for (int j = 0; j < NI; j++) acc[j] = f32x4_t{0, 0, 0, 0};
	for (int kf = w; kf < kfr; kf += 4 * U) {
		Frag a[U], b[U][NI];
#pragma unroll
		for (int u = 0; u < U; u++) {
			const int kc = min(kf + 4 * u, kfr - 1);
			a[u] = *reinterpret_cast<const Frag *>(A + (size_t)kc * TR::KF);
#pragma unroll
			for (int j = 0; j < NI; j++) b[u][j] = W[((size_t)min(n0 + j, nfr - 1) * kfr + kc) * 64];
		}
#pragma unroll
		for (int u = 0; u < U; u++) {
			if (kf + 4 * u >= kfr) a[u] = Frag{};
#pragma unroll
			for (int j = 0; j < NI; j++) acc[j] = TR::mma(b[u][j], a[u], acc[j]);
		}
	}
#pragma unroll
	for (int j = 0; j < NI; j++) s_acc[w][j][lane] = acc[j];
	__syncthreads();
	// wave w: column fragment w
	f32x4_t r;
#pragma unroll
	for (int e = 0; e < 4; e++) r[e] = (s_acc[0][w][lane][e] + s_acc[1][w][lane][e]) + (s_acc[2][w][lane][e] + s_acc[3][w][lane][e]);
	if (m0 + lr < g.M && n0 + w < nfr) tg_store4(g.C2 + (size_t)(m0 + lr) * g.ldc2 + (n0 + w) * 16 + 4 * lg, r);
}

// Few rows: a workgroup takes 16 MT rows x 16 NC columns of a part of K, its four waves a quarter of that each, and their sums meet
// in LDS.  The waves share no operand, so the loop has no barrier: a wave's weights come from memory in operand order, its rows as
// whole 128-byte lines that it turns in an LDS area of its own (as operands straight from memory, 16 rows of 64 bytes a load, they
// cost a unit four times as long: 130 rows x 10368 columns x K 1152 18.6 us).  FEW_AHEAD steps of 128 bytes of K are in flight;
// steps behind a wave's last are loads past the end of the buffers: zeros.
constexpr int FEW_AHEAD = 2, FEW_PITCH = 9;  // 16-byte pieces from row to row in LDS: operand reads meet every bank once
template <class TR, int EPI, int MT, int NC>
__global__ __launch_bounds__(256, 1) void linear_few_kernel(TgGemm g) {
	static_assert(EPI == TG_GE_F32 || EPI == TG_GE_GELU, "");
	typedef typename TR::T T;
	typedef typename TR::Frag Frag;
	constexpr int AREA = 16 * MT * FEW_PITCH;  // of a wave
	constexpr int SIZE = 4 * (AREA > MT * NC * 64 ? AREA : MT * NC * 64);
	__shared__ f32x4_t smem[SIZE];
	const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, lg = lane >> 4;
	const int nfr = g.N / 16, kfr = g.K / TR::KF, ntn = (nfr + NC - 1) / NC, ntm = (g.M + 16 * MT - 1) / (16 * MT);
	int b;
	{  // as in linear_kernel: a run of the tile order per XCD, so that a weight tile goes into one L2
		const int total = ntm * ntn * g.kparts, q = total >> 3, r = total & 7, x = (int)blockIdx.x & 7, i = (int)blockIdx.x >> 3;
		if (i >= q + (x < r ? 1 : 0)) return;
		b = x * q + min(x, r) + i;
	}
	const int part = b / (ntm * ntn);
	b -= part * ntm * ntn;
	const int tn = b / ntm, m0 = (b - tn * ntm) * 16 * MT;
	const int nst = kfr / 2, per = (nst + g.kparts - 1) / g.kparts, p0 = min(part * per, nst), n_part = min(per, nst - p0);
	const int k0 = p0 + n_part * w / 4, n = p0 + n_part * (w + 1) / 4 - k0;  // this wave's steps

	// views of this workgroup's rows and columns: offsets in them are below 4 GiB whatever the product's size
	const int rows_here = min(16 * MT, g.M - m0), cols_here = min(NC, nfr - tn * NC);
	const unsigned lda = (unsigned)(g.lda * (int)sizeof(T)), a_bytes = (unsigned)rows_here * lda, w_bytes = (unsigned)cols_here * (unsigned)kfr * 1024u;
	const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((unsigned char *)g.A + (size_t)m0 * lda, 0, a_bytes, 0x00020000);
	const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((unsigned char *)g.W + (size_t)tn * NC * kfr * 1024, 0, w_bytes, 0x00020000);
	unsigned ao[2 * MT], wo[NC];
#pragma unroll
	for (int i = 0; i < 2 * MT; i++) ao[i] = (unsigned)min(8 * i + (lane >> 3), rows_here - 1) * lda + (unsigned)(lane & 7) * 16u;
#pragma unroll
	for (int j = 0; j < NC; j++) wo[j] = (unsigned)min(j, cols_here - 1) * (unsigned)kfr * 1024u + (unsigned)lane * 16u;
	Frag fa[FEW_AHEAD][2 * MT], fb[FEW_AHEAD][2][NC];
	auto fetch = [&](int set, int s) {
		const unsigned sa = s < n ? (unsigned)(k0 + s) * 128u : a_bytes;
#pragma unroll
		for (int h = 0; h < 2; h++)
#pragma unroll
			for (int j = 0; j < NC; j++)
				fb[set][h][j] = __builtin_bit_cast(Frag, __builtin_amdgcn_raw_buffer_load_b128(rw, wo[j], s < n ? (unsigned)(2 * (k0 + s) + h) * 1024u : w_bytes, 0));
#pragma unroll
		for (int i = 0; i < 2 * MT; i++) fa[set][i] = __builtin_bit_cast(Frag, __builtin_amdgcn_raw_buffer_load_b128(ra, ao[i], sa, 0));
	};
	Frag *rows = reinterpret_cast<Frag *>(smem) + w * AREA;
	Frag *put = rows + (lane >> 3) * FEW_PITCH + (lane & 7), *get = rows + lr * FEW_PITCH + lg;
	f32x4_t acc[MT][NC];
#pragma unroll
	for (int i = 0; i < MT; i++)
#pragma unroll
		for (int j = 0; j < NC; j++) acc[i][j] = f32x4_t{0, 0, 0, 0};
#pragma unroll
	for (int d = 0; d < FEW_AHEAD; d++) fetch(d, d);
	for (int s = 0; s < n; s += FEW_AHEAD) {
#pragma unroll
		for (int d = 0; d < FEW_AHEAD; d++) {
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for (int i = 0; i < 2 * MT; i++) put[8 * i * FEW_PITCH] = fa[d][i];
#pragma unroll
			for (int h = 0; h < 2; h++)
#pragma unroll
				for (int i = 0; i < MT; i++) {
					const Frag a = get[16 * i * FEW_PITCH + 4 * h];
#pragma unroll
					for (int j = 0; j < NC; j++) acc[i][j] = TR::mma(fb[d][h][j], a, acc[i][j]);
				}
			__builtin_amdgcn_sched_barrier(0);
			fetch(d, s + d + FEW_AHEAD);
		}
	}
	__syncthreads();
	f32x4_t(*s_acc)[MT * NC][64] = reinterpret_cast<f32x4_t(*)[MT * NC][64]>(smem);
#pragma unroll
	for (int i = 0; i < MT; i++)
#pragma unroll
		for (int j = 0; j < NC; j++) s_acc[w][i * NC + j][lane] = acc[i][j];
	__syncthreads();
	// lane: row lr, columns 4 lg ... of tile (i, j)
	for (int t = w; t < MT * NC; t += 4) {
		const int i = t / NC, m = m0 + 16 * i + lr, at = (tn * NC + t - i * NC) * 16 + 4 * lg;
		f32x4_t r;
#pragma unroll
		for (int e = 0; e < 4; e++) r[e] = (s_acc[0][t][lane][e] + s_acc[1][t][lane][e]) + (s_acc[2][t][lane][e] + s_acc[3][t][lane][e]);
		if (m >= g.M || at >= g.N) continue;
		if (EPI == TG_GE_GELU) {
#pragma unroll
			for (int e = 0; e < 4; e++) r[e] = tg_gelu(r[e]);
			tg_store4((T *)g.C + (size_t)m * g.ldc + at, r);
		} else {
			tg_store4(g.C2 + (size_t)part * g.part_stride + (size_t)m * g.ldc2 + at, r);
		}
	}
}

// 128-row tiles where they fill the device's 512 places (two workgroups per compute unit), then 64 rows, then 32
bool linear_rows32(int rows, int ntn) { return (rows + 127) / 128 * ntn < 448 && (rows + 63) / 64 * ntn < 256; }

// A product of few rows has few tiles, and each walks all of K at the pace of one workgroup on an otherwise idle compute unit
// (0.33 us a stage of 128 bytes of K: 53 us for 130 rows x 1152 columns x K 10368 in 45 workgroups).  Its K is cut until the parts
// fill the 512 places or are down to TG_LINEAR_PART_STAGES stages, whose start-up and sums would cost more than they save.  A
// Tutelix prompt of 600 tokens in portions of 130 (width 1152, 26 layer runs) with 24 steps behind it: 51.0 -> 45.8 ms.
constexpr int TG_LINEAR_PART_STAGES = 12;
int linear_tile_parts(int rows, int N, int K, int dt) {
	const int ntn = (N + 127) / 128, stages = K * (int)tg_dt_bytes(dt) / 128;
	if (!linear_rows32(rows, ntn)) return 1;
	const int tiles = (rows + 31) / 32 * ntn;
	int p = 1;
	while (p < 8 && 2 * p * tiles <= 512 && stages / (2 * p) >= TG_LINEAR_PART_STAGES) p *= 2;
	return p;
}

// Whether a product that the tiles above would cut into 32 rows runs in linear_few_kernel instead, in which of its instances and, where
// the consumer can add parts of K, in how many.  Times follow a count of steps of K times rounds of 256 workgroups (0.045 us a unit
// and 2.5 us for the launch, the first loads and the sums): MT + NC units a step in bf16 (a unit's path to its L1), 1.1 MT NC in fp32
// (the matrix instructions), 8 and 14 of a 32-row tile; a part costs its way through memory once more.  Measured, us, tiles against
// the choice here: 130 rows, width 1152, feed-forward 10368: up 17.1 and 13.8 (3 x 4), down 17.8 in 8 parts and 13.7 in 4, mixer
// output 7.1 and 4.1 (3 x 2 in 2); 9 rows: 10.3 and 8.0, 10.8 and 7.2 (1 x 4); 333 rows, width 640: mixer output in fp32 11.9 and
// 5.3 (1 x 2), down in bf16 7.9 and 6.4 (2 x 4 in 2); 20 rows, fp32: 14.4 and 5.5, 12.9 and 4.8.
// Only for sums that depend on the number of rows already: products in parts of K, and, in models whose down projections are
// (width above 256), the one in front of those.  The others keep one order of sums, so that a prompt's rows are the same bits
// however long it goes on.
bool linear_split_sums(int width) { return width > 256; }
struct LinearFew {
	int mt, nc, parts;  // mt 0: the tiles
};
LinearFew linear_few(int rows, int N, int K, int dt, bool can_part) {
	const int ntn = (N + 127) / 128, stages = K * (int)tg_dt_bytes(dt) / 128;
	LinearFew best = {0, 0, 1};
	if (!linear_rows32(rows, ntn)) return best;
	auto rounds = [](long long wgs) { return (wgs + 255) / 256; };
	// costs in 1/32 units; a part's 8 bytes an element at 4 TB/s
	auto cost_of = [&](long long wgs, int parts, int step) {
		return rounds(wgs * parts) * ((stages + parts - 1) / parts) * step + (parts > 1 ? (long long)parts * rows * N / 710 : 0);
	};
	const int tile_parts = can_part ? linear_tile_parts(rows, N, K, dt) : 1;
	long long least = cost_of((long long)((rows + 31) / 32) * ntn, tile_parts, 32 * (dt == TG_DT_BF16 ? 8 : 14));
	static const int shapes[][2] = {{1, 2}, {1, 4}, {2, 4}, {3, 2}, {3, 4}};
	for (const auto &t : shapes)
		for (int parts = 1; parts <= (can_part ? 8 : 1) && (parts == 1 || stages / parts >= 4); parts *= 2) {
			const long long wgs = (long long)((rows + 16 * t[0] - 1) / (16 * t[0])) * ((N / 16 + t[1] - 1) / t[1]);
			const long long c = cost_of(wgs, parts, dt == TG_DT_BF16 ? 32 * (t[0] + t[1]) : 36 * t[0] * t[1]);
			if (c < least) {
				least = c;
				best = {t[0], t[1], parts};
			}
		}
	return best;
}

template <class TR, int EPI>
bool launch_few(const TgGemm &g, hipStream_t s) {
	if (EPI == TG_GE_GELU ? !linear_split_sums(g.K) : g.kparts < 1) return false;
	const LinearFew f = linear_few(g.M, g.N, g.K, TR::DT, EPI == TG_GE_F32);
	if (f.mt == 0) return false;
	TgGemm p = g;
	p.kparts = f.parts;
	const dim3 grid((unsigned)((g.N / 16 + f.nc - 1) / f.nc * ((g.M + 16 * f.mt - 1) / (16 * f.mt)) * f.parts + 7));  // (a run per XCD)
	auto go = [&](auto *kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, p); };
	if (f.mt == 1 && f.nc == 2) go(linear_few_kernel<TR, EPI, 1, 2>);
	else if (f.mt == 1) go(linear_few_kernel<TR, EPI, 1, 4>);
	else if (f.mt == 2) go(linear_few_kernel<TR, EPI, 2, 4>);
	else if (f.nc == 2) go(linear_few_kernel<TR, EPI, 3, 2>);
	else go(linear_few_kernel<TR, EPI, 3, 4>);
	return true;
}

template <class TR, int EPI>
void launch_linear_t(const TgGemm &g, hipStream_t s) {
	if constexpr (EPI == TG_GE_F32) {
		if (g.N <= 256) {
			hipLaunchKernelGGL((linear_thin_kernel<TR>), dim3((unsigned)((g.M + 15) / 16), (unsigned)((g.N + 63) / 64)), dim3(256), 0, s, g);
			return;
		}
	}
	if (g.tiles) {
		if constexpr (EPI == TG_GE_STORE || EPI == TG_GE_SWIGLU) {
			const unsigned grid = (unsigned)g.max_tiles * (unsigned)((g.N + 127) / 128);
			if (g.tile_rows == 128)
				hipLaunchKernelGGL((linear_kernel<TR, EPI, 2, 2, 4, 4, true>), dim3(grid), dim3(256), 0, s, g);
			else if (g.tile_rows == 64)
				hipLaunchKernelGGL((linear_kernel<TR, EPI, 2, 2, 2, 4, true>), dim3(grid), dim3(256), 0, s, g);
			else
				hipLaunchKernelGGL((linear_kernel<TR, EPI, 1, 4, 2, 2, true>), dim3(grid), dim3(256), 0, s, g);
		}
		return;
	}
	if constexpr (EPI == TG_GE_F32 || EPI == TG_GE_GELU) {
		if (launch_few<TR, EPI>(g, s)) return;
	}
	const int ntn = (g.N + 127) / 128, rows = EPI == TG_GE_TRANS ? g.rows_out : g.M;
	if constexpr (EPI == TG_GE_F32) {
		TgGemm p = g;
		p.kparts = g.kparts > 1 ? g.kparts : 1;
		if (linear_rows32(rows, ntn)) {
			hipLaunchKernelGGL((linear_kernel<TR, EPI, 1, 4, 2, 2, false>), dim3((unsigned)((rows + 31) / 32 * ntn * p.kparts)), dim3(256), 0, s, p);
			return;
		}
	}
	const int t128 = (rows + 127) / 128 * ntn, t64 = (rows + 63) / 64 * ntn;
	if (t128 >= 448)
		hipLaunchKernelGGL((linear_kernel<TR, EPI, 2, 2, 4, 4, false>), dim3((unsigned)((rows + 127) / 128 * ntn)), dim3(256), 0, s, g);
	else if (!linear_rows32(rows, ntn))
		hipLaunchKernelGGL((linear_kernel<TR, EPI, 2, 2, 2, 4, false>), dim3((unsigned)t64), dim3(256), 0, s, g);
	else
		hipLaunchKernelGGL((linear_kernel<TR, EPI, 1, 4, 2, 2, false>), dim3((unsigned)((rows + 31) / 32 * ntn)), dim3(256), 0, s, g);
}

template <class TR>
void launch_linear_dt(const TgGemm &g, int epi, hipStream_t s) {
	switch (epi) {
		case TG_GE_STORE: launch_linear_t<TR, TG_GE_STORE>(g, s); break;
		case TG_GE_F32: launch_linear_t<TR, TG_GE_F32>(g, s); break;
		case TG_GE_RESID: launch_linear_t<TR, TG_GE_RESID>(g, s); break;
		case TG_GE_GELU: launch_linear_t<TR, TG_GE_GELU>(g, s); break;
		case TG_GE_SWIGLU: launch_linear_t<TR, TG_GE_SWIGLU>(g, s); break;
		default: launch_linear_t<TR, TG_GE_TRANS>(g, s); break;
	}
}

unsigned pack_grid(const TgPack &p) {
	const long long n = ((long long)p.rows * p.cols + 255) / 256;
	return (unsigned)(n < 16384 ? (n > 0 ? n : 1) : 16384);
}

}  // namespace

void tg_launch_pack(const TgMat &dst, int dt, const TgPack &p, hipStream_t s) {
	if (dt == TG_DT_BF16) hipLaunchKernelGGL((pack_kernel<TgB16>), dim3(pack_grid(p)), dim3(256), 0, s, (__bf16 *)dst.w, dst.k, p);
	else hipLaunchKernelGGL((pack_kernel<TgF32>), dim3(pack_grid(p)), dim3(256), 0, s, (float *)dst.w, dst.k, p);
}

void tg_launch_unpack_f32(float *dst, int ld, const TgPack &p, hipStream_t s) {
	hipLaunchKernelGGL(unpack_f32_kernel, dim3(pack_grid(p)), dim3(256), 0, s, dst, ld, p);
}

int tg_vec_blocks(const TgVec &v, int epi) {
	if (vec_wide(v, epi)) return (v.ntiles + 3) / 4;
	return epi == TG_VE_SWIGLU || vec_pairs(v, epi) ? (v.ntiles + 1) / 2 : v.ntiles;
}

// Parts of K for a product whose consumer adds them: two workgroups per compute unit, at least 8 fragments per part (up to one
// workgroup per unit only, a down projection of 24 MB left a quarter of the units with two of 288: Tutelix 1152, 600 tokens and 24
// steps 43.3 -> 42.7 ms).
int tg_vec_ksplit(int ntiles, int nz, int kfrags, int n_cu) {
	int p = 1;
	while (p < 8 && ntiles * nz * p < 2 * n_cu && kfrags / (2 * p) >= 8) p *= 2;
	return p;
}

void tg_launch_vec(const TgVec &v, int dt, int pro, int epi, hipStream_t s) {
	if (dt == TG_DT_BF16) launch_vec_dt<TgB16>(v, pro, epi, s);
	else launch_vec_dt<TgF32>(v, pro, epi, s);
}

int tg_linear_kparts(int rows, int N, int K, int dt) {
	if (!linear_split_sums(N)) return 1;
	const LinearFew f = linear_few(rows, N, K, dt, true);
	return f.mt ? f.parts : linear_tile_parts(rows, N, K, dt);
}

void tg_launch_linear(const TgGemm &g, int dt, int epi, hipStream_t s) {
	if (dt == TG_DT_BF16) launch_linear_dt<TgB16>(g, epi, s);
	else launch_linear_dt<TgF32>(g, epi, s);
}
