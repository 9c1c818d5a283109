// The layers of a Gemma decode step as ONE launch of resident workgroups that hand over inside an XCD wherever they can
// (transformer.hpp:75-97 of the reference: the layer loop of forward_decode; modules.hpp:135-220: what a layer does).
//
// What bounds a step is its chain of dependent products, not its bytes: one launch per product costs 4.3 us each (2.5 us
// between dependent launches, then inputs, weights and reductions in turn), five of them a layer.  Measured on this part, with
// 32 units per XCD: a hand-over between all 256 compute units through memory costs 1.0 us when a unit reads only the values it
// owns, one among the units of an XCD through their shared L2 0.7 us (all of 1152 words, read by everybody).  So the work is
// cut by XCD:
//
//   * XCD x computes query head x / 2 and attends to half x % 2 of the keys, and multiplies the result by the head's 256
//     rows of the output projection; it owns an eighth of the feed-forward, columns of up and gate and the same rows of
//     down.  Q|K|V -> attention -> output projection and up|gate -> down are hand-overs inside the XCD.
//   * What crosses the XCDs are their eight partial sums of a layer's two outputs: compute unit r of every XCD adds up
//     columns r * H / 32 ... of the eight, and hands its sums to the 32 units of its own XCD, which all need the whole vector.
//
// A step of the 1B shape behind 178 tokens takes 419 us (608 with one launch per product), of the 270m shape behind 64 tokens
// 208 us (326), the head's launch of 50 and 30 us included: 14 and 9.5 us a layer against 21.5 and 16.  Contexts of 31,000
// tokens: 570 (678) and 327 us (389).
//
// A wave is an actor of its own with one or two roles (product tile, attention, sums); there is no barrier in the layer
// loop.  Waves poll the data themselves: a slot of the exchange buffer holds a pattern no result has (a NaN; results that
// are this NaN are stored as another) until its value arrives.  Slots come in a ring of four layers; their writer resets
// them two layers later, when every reader has long delivered something this layer depends on, and a reader that meets the
// slot again has seen the writer's value of the layer before, which the writer stored behind the acknowledged reset.
//   - Values for the own XCD are stored plainly: they stop at the XCD's L2, and loads at device scope, which skip the L1,
//     find them there.  Values for other XCDs are stored and loaded at device scope.
//   - Polling loads the L2 that the values pass through: with every waiting wave at it a layer of the 270m shape took 12.2 us
//     instead of 10.  A wave that waits for long waits for a counter in LDS first, which its own workgroup's producer moves.
//   - Every wait is bounded: a wave that polls max_spins times in vain writes the step's token and position to the error
//     block and leaves; the others see the word or their own bound, launches that follow return at once, and the host
//     repeats the steps with one launch per product.
//
// Products run on the matrix cores with int8 weights as they are and the input row as four signed base-256 digits of a
// 30-bit fixed point number (largest magnitude of the row; of the XCD's slice for the down projection): the four digit rows
// are four of the 16 rows of v_mfma_i32_16x16x64_i8, the products and sums are exact, and no lane reduction follows.  The
// rounding of the row is 2^-30 of its largest value, against 2^-24 of every partial sum in a chain of fp32 additions.  A tile
// of 16 columns over the whole K belongs to one wave, which holds its weights in registers: they are requested a layer
// ahead, at a place that has no wait of the wave's close behind it (a wait for a poll also waits for every load issued
// before).  The weights are those of the prefill products ([K/16][128 columns][16 rows]): a lane's 16 bytes are its operand.
// (Measured and not taken: products in waves of their own that never poll, fed with digits through LDS by two waves that hold
// the stream: 212 and 430 us, the counters between the two cost 0.3 us a product.)

#include "tg_attn_decode.h"
#include "tg_gemv_parts.h"
#include "tg_internal.h"

using namespace tgp;

namespace {

constexpr int RNT = 512;      // eight waves, one workgroup per compute unit (its registers allow no second one)
constexpr int RX = 8, RU = 32;  // XCDs, compute units of one
constexpr unsigned SENTINEL = 0xffffffffu;
constexpr int AUX_DEV = 16;   // sc1: device scope
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int plane_stride(int k) {  // dwords of one digit plane: four planes start 16 banks apart
	int p = k / 4;
	while (p % 64 != 16) p++;
	return p;
}

template <int H, int F>
struct Geo {
	static constexpr int W = H / RU;                 // output columns of a compute unit
	static constexpr int CT = (W + 15) / 16;         // ... in tiles of 16
	static constexpr int NQ = (H / 4 + 63) / 64;     // 16-byte pieces of the residual stream per lane
	static constexpr int KSH = H / 64;               // steps of 64 rows over the residual stream
	static constexpr int PAIRS = F / (RX * RU);      // up|gate pairs of a compute unit
	static constexpr int UGT = (PAIRS + 7) / 8;      // ... in tiles of eight pairs
	static constexpr int KD = F / RX;                // rows of the down projection of an XCD
	static constexpr int KSD = (KD + 63) / 64, KDP = KSD * 64, NQD = (KD / 4 + 63) / 64;
	static constexpr int PSH = plane_stride(H), PSD = plane_stride(KDP), PSO = plane_stride(256);
	static constexpr int PSM = PSH > PSD ? PSH : PSD;  // dwords of a plane in a wave's scratch (PSO is smaller: H >= 256)
	static_assert(H % 128 == 0 && (UGT < 4 || CT < 4) && F % (RX * RU) == 0 && KD % 16 == 0 && CT <= 3 && UGT <= 4 && H / 4 % 32 == 0, "widths this split covers");
	// one layer's part of the exchange buffer, in words
	static constexpr int XO = 0, XD = RX * H, XML = 2 * RX * H, LOC = XML + RX * 32;
	static constexpr int PO = 0, PD = H, QKV = 2 * H, AP = QKV + 768, AML = AP + RU * 256, HB = AML + 2 * RU, LOCN = HB + KDP;
	static constexpr int SLOT = LOC + RX * LOCN;
};

__device__ __forceinline__ unsigned not_sentinel(float v) {
	const unsigned b = __float_as_uint(v);
	return b == SENTINEL ? 0x7fc00000u : b;
}
__device__ __forceinline__ unsigned max4(u32x4 v) { return max(max(v[0], v[1]), max(v[2], v[3])); }

// What a wait needs.
struct Wait {
	unsigned *err;
	int max_spins, tok, pos, step;
	bool pending;  // the launch was to record the pick of the step before
	__device__ __forceinline__ bool again(int &spins) const {  // false: give up
		if (++spins >= max_spins) {
			if ((threadIdx.x & 63) == 0) {
				err[1] = (unsigned)tok;
				err[2] = (unsigned)pos;
				err[3] = (unsigned)step;
				err[4] = pending ? 1u : 0u;
				__hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			}
			return false;
		}
		// (read as a scalar: a condition per lane would make every address behind the wait one)
		if ((spins & 255) == 0 && __builtin_amdgcn_readfirstlane((int)__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0) return false;
		__builtin_amdgcn_s_sleep(1);
		asm volatile("" ::: "memory");
		return true;
	}
};

// A counter of the own workgroup in LDS that reaches `target` when a value polled for next is about to be complete: waves that
// wait for long do not load the L2 meanwhile.
__device__ __forceinline__ bool wait_near(const unsigned *flag, unsigned target, const Wait &wt) {
	int spins = 0;
	while ((int)(__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) - target) < 0)
		if (!wt.again(spins)) return false;
	return true;
}
__device__ __forceinline__ void signal_near(unsigned *flag) {
	if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_add(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The pieces lane, lane + 64, ... of 16 bytes of a view (past its end: zeros, without a memory access); false once the wait has
// given up
template <int N>
__device__ __forceinline__ bool poll_row(u32x4 (&v)[N], const __amdgpu_buffer_rsrc_t r, const Wait &wt) {
	const unsigned voff = (threadIdx.x & 63) * 16u;
	int spins = 0;
	for (;;) {
#pragma unroll
		for (int i = 0; i < N; i++) v[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff + 1024u * (unsigned)i, 0, AUX_DEV));
		unsigned m = 0;
#pragma unroll
		for (int i = 0; i < N; i++) m = max(m, max4(v[i]));
		if (__all(m != SENTINEL)) return true;
		if (!wt.again(spins)) return false;
	}
}
// The word at voff of N rows that lie `step` bytes apart
template <int N>
__device__ __forceinline__ bool poll_column(unsigned (&v)[N], const __amdgpu_buffer_rsrc_t r, unsigned voff, unsigned step, const Wait &wt) {
	int spins = 0;
	for (;;) {
#pragma unroll
		for (int i = 0; i < N; i++) v[i] = __builtin_amdgcn_raw_buffer_load_b32(r, voff, step * (unsigned)i, AUX_DEV);
		unsigned m = 0;
#pragma unroll
		for (int i = 0; i < N; i++) m = max(m, v[i]);
		if (__all(m != SENTINEL)) return true;
		if (!wt.again(spins)) return false;
	}
}

// KS steps of 64 rows of a tile of 16 columns: step u's pieces are 4 * 2048 bytes behind those of the step before.  A pause of
// 192 clocks in front of each: the polls and stores of a hand-over wait behind whatever a compute unit, and the fabric, have
// been asked for.  Microseconds of a step of the 1B shape: 458 when the feed-forward's tiles are requested in one burst behind
// the down product, 446 with pauses there, 425 with the up|gate tiles only behind the next layer's Q, 419 with both there (the
// 270m shape, whose weights come from the memory-side cache, 204 to 206 in all forms).
template <int KS>
__device__ __forceinline__ void load_tile(i32x4 (&b)[KS], const int8_t *W, uint32_t bytes, uint32_t voff) {
	const __amdgpu_buffer_rsrc_t r = make_rsrc(W, bytes);
#pragma unroll
	for (int u = 0; u < KS; u++) {
		if (KS > 4) {
			__builtin_amdgcn_s_sleep(3);
			asm volatile("" ::: "memory");
		}
		b[u] = ldw<TG_W_DEFAULT>(r, voff, min((uint32_t)u * 8192u, bytes));  // never past the records: their difference is unsigned
	}
}

// The digits of one 16-byte piece (four rows of K) into a wave's scratch.
__device__ __forceinline__ void put_digits(unsigned *dg, int stride, int piece, const float *u, float mul) {
	unsigned d[4];
	tg_quant4<4>(u, mul, d);
#pragma unroll
	for (int p = 0; p < 4; p++) dg[p * stride + piece] = d[p];
}
// Columns' sums of a tile as floats, in lanes 0 .. 15 (the digit rows 0 .. 3 of the result are the four registers there).
template <int KS>
__device__ __forceinline__ float tile_product(const i32x4 (&b)[KS], const unsigned *dg, int stride) {
	const int lane = threadIdx.x & 63;
	const unsigned *src = dg + (lane & 3) * stride + 4 * (lane >> 4);
	i32x4 acc = i32x4{0, 0, 0, 0}, acc2 = acc;  // two chains: an instruction takes longer than the next may start behind it
	constexpr int D = KS < 6 ? KS : 6;  // operands read ahead (all of them at once cost the registers the weights are in)
	i32x4 a[D];
#pragma unroll
	for (int u = 0; u < D; u++) a[u] = *reinterpret_cast<const i32x4 *>(src + 16 * u);
#pragma unroll
	for (int u = 0; u < KS; u++) {
		if (u & 1) acc2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u % D], b[u], acc2, 0, 0, 0);
		else acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u % D], b[u], acc, 0, 0, 0);
		if (u + D < KS) a[u % D] = *reinterpret_cast<const i32x4 *>(src + 16 * (u + D));
		__builtin_amdgcn_sched_barrier(0);
	}
	acc += acc2;
	return fmaf(fmaf(fmaf((float)acc[3], 256.0f, (float)acc[2]), 256.0f, (float)acc[1]), 256.0f, (float)acc[0]);
}
// Scale of a row from the bits of its largest magnitude; a row that holds an infinity or a NaN gives NaNs.
__device__ __forceinline__ float digit_factors(unsigned maxbits, float &mul) {
	float inv;
	tg_row_factors<4>(__uint_as_float(maxbits), mul, inv);
	return maxbits >= 0x7f800000u ? __uint_as_float(0x7fc00000u) : inv;
}
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
	v = max(v, tg_red_partner_u32<32>(v));
	v = max(v, tg_red_partner_u32<16>(v));
	v = max(v, tg_red_partner_u32<8>(v));
	v = max(v, tg_red_partner_u32<4>(v));
	v = max(v, tg_red_partner_u32<2>(v));
	v = max(v, tg_red_partner_u32<1>(v));
	return v;
}

// The residual stream, held by every wave that computes norms: lane l owns the pieces l, l + 64, ... of four elements.  Pieces
// past the end are 0 in the stream, in block outputs and in norm weights (the end of a buffer view), and their digits fall
// between the planes.
template <int H, int NQ>
struct Stream {
	f32x4 r[NQ];
	static __device__ __forceinline__ void load(f32x4 (&w)[NQ], const float *src) {
		const __amdgpu_buffer_rsrc_t rs = make_rsrc(src, H * 4u);
#pragma unroll
		for (int i = 0; i < NQ; i++) w[i] = ldx(rs, (threadIdx.x & 63) * 16u + 1024u * (unsigned)i, 0);
	}
	// norm weights kept in a wave's LDS while it waits: [NQ][64 lanes]
	static __device__ __forceinline__ void park(f32x4 *dst, const float *src) {
		f32x4 w[NQ];
		load(w, src);
#pragma unroll
		for (int i = 0; i < NQ; i++) dst[(threadIdx.x & 63) + 64 * i] = w[i];
	}
	static __device__ __forceinline__ void unpark(f32x4 (&w)[NQ], const f32x4 *src) {
#pragma unroll
		for (int i = 0; i < NQ; i++) w[i] = src[(threadIdx.x & 63) + 64 * i];
	}
	// modules.hpp:166-168 / 218-219: x = rmsnorm(block output, post) + x
	__device__ __forceinline__ void add_post_norm(const u32x4 (&pv)[NQ], const f32x4 (&wpo)[NQ]) {
		__builtin_amdgcn_sched_barrier(0);
		float ss = 0.0f;
#pragma unroll
		for (int i = 0; i < NQ; i++)
#pragma unroll
			for (int e = 0; e < 4; e++) ss = fmaf(__uint_as_float(pv[i][e]), __uint_as_float(pv[i][e]), ss);
		const float irms = rms_inv(wave_sum(ss), H);
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int i = 0; i < NQ; i++)
#pragma unroll
			for (int e = 0; e < 4; e++) r[i][e] = (__uint_as_float(pv[i][e]) * irms) * (wpo[i][e] + 1.0f) + r[i][e];
	}
	// ops.hpp:126-180: the digits of x * (1 + w) into a wave's scratch; returns what the integer sums are multiplied by
	__device__ __forceinline__ float pre_norm_digits(const f32x4 (&wpre)[NQ], unsigned *dg, int stride) const {
		__builtin_amdgcn_sched_barrier(0);
		float ss = 0.0f;
		unsigned mb = 0;
		float u[NQ][4];
#pragma unroll
		for (int i = 0; i < NQ; i++)
#pragma unroll
			for (int e = 0; e < 4; e++) {
				ss = fmaf(r[i][e], r[i][e], ss);
				u[i][e] = r[i][e] * (wpre[i][e] + 1.0f);
				mb = max(mb, __float_as_uint(u[i][e]) & 0x7fffffffu);
			}
		const float irms = rms_inv(wave_sum(ss), H);
		float mul;
		const float inv = digit_factors(wave_max_u32(mb), mul);
#pragma unroll
		for (int i = 0; i < NQ; i++) {
			__builtin_amdgcn_sched_barrier(0);  // (piece by piece: in flight together they push weights out of the registers)
			put_digits(dg, stride, (int)(threadIdx.x & 63) + 64 * i, u[i], mul);
		}
		__builtin_amdgcn_sched_barrier(0);
		return inv * irms;
	}
	__device__ __forceinline__ void store(float *dst) const {
		const __amdgpu_buffer_rsrc_t rs = make_rsrc(dst, H * 4u);  // (a store past the end is dropped)
#pragma unroll
		for (int i = 0; i < NQ; i++) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, r[i]), rs, (threadIdx.x & 63) * 16u + 1024u * (unsigned)i, 0, 0);
	}
	__device__ __forceinline__ void embed(const TgResident &f, int tok) {  // ops.hpp:537-568
		f32x4 s[NQ];
		load(s, f.wte_scales);
		const int8_t *row = f.wte + (size_t)tok * H;
#pragma unroll
		for (int i = 0; i < NQ; i++) {
			const int q4 = *reinterpret_cast<const int *>(row + 4 * min((int)(threadIdx.x & 63) + 64 * i, H / 4 - 1));
#pragma unroll
			for (int e = 0; e < 4; e++) r[i][e] = embed_value(s[i][e], f.emb_scale, (int8_t)(q4 >> (8 * e)));
		}
	}
};

// Keys of a layer that an XCD attends to, and how they are dealt: blocks of eight keys, two waves of a compute unit take one
// each.  Up to 32 blocks (256 keys of the half: a full window of 512) go to every other unit, so that the results to be
// merged are few; more keys go to all units, and waves walk their blocks.
constexpr int AW = 2;  // attention waves of a compute unit
struct Keys {
	int first, n, cur, parts, part;  // first slot, slots, slot of this token; results to merge, the unit's own (or -1)
	int max_pos;                     // slots of the cache
	bool mine;                       // the token's own slot is among them
	__device__ __forceinline__ Keys(int pos, int bp, int slots, int x, int rank) : max_pos(slots) {
		const int valid = min(pos + 1, max_pos), half = (valid + 1) >> 1;
		cur = bp % max_pos;
		first = (x & 1) ? half : 0;
		n = (x & 1) ? valid - half : half;
		mine = cur >= first && cur < first + n;
		const int blocks = (n + 7) >> 3;
		const bool few = blocks <= AW * RU / 2;
		parts = max(1, min(RU, (blocks + AW - 1) / AW));
		part = few ? ((rank & 1) == 0 ? rank >> 1 : -1) : rank;
		if (part >= parts) part = -1;
	}
};

// Greedy pick of the previous step from its head's pairs (see argmax_pairs), by all threads of the workgroup.
__device__ __forceinline__ int pick_of_pairs(const float *val, const int *idx, int n, float *s_bv, int *s_bi) {
	const int tid = threadIdx.x;
	float bv = -INFINITY;
	int bi = 0x7fffffff;
	for (int i0 = 0; i0 < n; i0 += 4 * RNT) {
		float ov[4];
		int oi[4];
#pragma unroll
		for (int u = 0; u < 4; u++) {
			const int i = min(i0 + u * RNT + tid, n - 1);
			ov[u] = val[i];
			oi[u] = idx[i];
		}
#pragma unroll
		for (int u = 0; u < 4; u++)
			if (ov[u] > bv || (ov[u] == bv && oi[u] < bi)) { bv = ov[u]; bi = oi[u]; }  // (a pair met twice changes nothing)
	}
#define TG_STEP(O)                                                      \
	{                                                                   \
		const float ov = tg_red_partner<O>(bv);                         \
		const int oi = tg_red_partner<O>(bi);                           \
		if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }     \
	}
	TG_STEP(32) TG_STEP(16) TG_STEP(8) TG_STEP(4) TG_STEP(2) TG_STEP(1)
#undef TG_STEP
	if ((tid & 63) == 0) { s_bv[tid >> 6] = bv; s_bi[tid >> 6] = bi; }
	__syncthreads();
	bv = s_bv[0];
	bi = s_bi[0];
	for (int i = 1; i < RNT / 64; i++)
		if (s_bv[i] > bv || (s_bv[i] == bv && s_bi[i] < bi)) { bv = s_bv[i]; bi = s_bi[i]; }
	return bi == 0x7fffffff ? -1 : bi;
}

template <int H, int F>
__global__ __launch_bounds__(RNT) void decode_resident_kernel(const TgResident f) {
	using G = Geo<H, F>;
	using S = Stream<H, G::NQ>;
	__shared__ __attribute__((aligned(16))) unsigned dg_s[RNT / 64][4 * G::PSM];
	__shared__ f32x4 norm_s[G::UGT + 2][2][64 * G::NQ];  // of the up|gate waves and of waves 4 and 5
	__shared__ __attribute__((aligned(16))) float lut_s[LUT_LDS];
	__shared__ __attribute__((aligned(16))) float pacc[AW][256];
	__shared__ float pm[AW], pl[AW];
	__shared__ unsigned arrived;
	__shared__ unsigned near_q, near_o, near_po, near_d, near_pd;  // see wait_near: Q, output projection, its sums, down, its sums
	__shared__ float s_bv[RNT / 64];
	__shared__ int s_bi[RNT / 64];

	const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
	int xcc;
	asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(xcc));
	const int x = __builtin_amdgcn_readfirstlane(xcc) & 7, rank = (int)(blockIdx.x >> 3);  // workgroups are dealt to the XCDs in turn (checked by the host once)
	const int col = lane & 15, kq = lane >> 4;             // a lane's column of a tile and its 16 of the 64 rows of a step
	unsigned *dg = dg_s[w];

	// ---- the token, the table of the gated product ----
	if (tid == 0) arrived = near_q = near_o = near_po = near_d = near_pd = 0;
	const bool lut_in_lds = f.lut_size <= LUT_LDS;
	if (lut_in_lds)
		for (int i = tid; i < f.lut_size; i += RNT) lut_s[i] = f.lut[i];
	const unsigned dead = __hip_atomic_load(f.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	int tok;
	if (f.am_val != nullptr) tok = pick_of_pairs(f.am_val, f.am_idx, f.am_n, s_bv, s_bi);
	else tok = *f.tok;
	if (__syncthreads_or(dead != 0u)) return;
	if (f.am_val != nullptr && blockIdx.x == 0 && tid == 0) record_pick(tok, f.am_ctr, f.am_log, 1);
	const int raw_tok = tok;
	tok = __builtin_amdgcn_readfirstlane(tok < 0 ? 0 : (tok >= f.vocab ? f.vocab - 1 : tok));
	const Wait wt{f.err, f.max_spins, raw_tok, f.pos, f.step, f.am_val != nullptr};

	// the table of the layers' pointers is read through the constant address space: behind a store or a wait the compiler would
	// fetch it with vector loads otherwise, pointers in vector registers and all that follows from it
	typedef const TgResidentLayer __attribute__((address_space(4))) *Table;
	const Table tab = (Table)f.layers;
	auto slot_of = [&](int l) { return f.xch + (size_t)((f.ring + l) & 3) * G::SLOT; };
	auto local_of = [&](int l) { return slot_of(l) + G::LOC + (size_t)x * G::LOCN; };
	auto local_view = [&](int l, int word, int n) { return make_rsrc(local_of(l) + word, (uint32_t)n * 4u); };
	auto cross_view = [&](int l, int word, int n) { return make_rsrc(slot_of(l) + word, (uint32_t)n * 4u); };
	auto store_local = [&](int l, int word, float v) { __hip_atomic_store(local_of(l) + word, not_sentinel(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
	auto store_dev = [&](int l, int word, unsigned bits) { __hip_atomic_store(slot_of(l) + word, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
	// the slot of layer l + 2 is that of layer l - 2 as well: what this wave stored there is reset (the last two layers' by the next step)
	auto reset_local = [&](int l, int word) { __hip_atomic_store(local_of(l + 2) + word, SENTINEL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
	const uint32_t bytes_h = (uint32_t)H * (uint32_t)(4 * 256 + 512), bytes_o = 1024u * (uint32_t)H, bytes_ug = 2u * (uint32_t)H * (uint32_t)F,
	               bytes_d = (uint32_t)F * (uint32_t)H;
	// byte offset of a lane's first piece: virtual column c, first row 16 * k16 of a matrix of K rows
	auto piece_at = [&](int c, int k16, int K) { return (uint32_t)(((c >> 7) * (K >> 4) + k16) * 2048 + (c & 127) * 16); };
	const int ocol = [&] {  // a lane's output column of tile t is ocol + 16 t, of the last tile its valid ones
		return rank * G::W;
	}();
	auto out_col = [&](int t) { return ocol + 16 * t + min(col, min(16, G::W - 16 * t) - 1); };

	if (w < 4) {
		// ================ up|gate tile w, down tile w, sums of the XCDs' partial outputs (wave 3) ================
		const bool ug = w < G::UGT, dn = w < G::CT, red = w == 3;
		if (!ug && !dn && !red) return;
		S st;
		i32x4 bu[G::KSH], bd[G::KSD];
		float su = 0.0f, sd = 0.0f;
		const int np = min(8, G::PAIRS - 8 * w);  // pairs of the tile (of a wave without one: unused)
		const int pair = x * G::KD + rank * G::PAIRS + 8 * w + min(col & 7, max(np, 1) - 1);
		const int ugcol = ug ? (pair >> 6) * 128 + (pair & 63) + ((col & 8) ? 64 : 0) : 0;
		const uint32_t ug_off = piece_at(ugcol, kq, H);
		const int dcol = dn ? out_col(w) : 0;
		const uint32_t d_off = piece_at(dcol, x * (G::KD / 16) + kq, F);
		auto issue_ug = [&](int l) {
			load_tile<G::KSH>(bu, tab[l].Wug, bytes_ug, ug_off);
			su = tab[l].sug[ugcol];
		};
		auto issue_d = [&](int l) {
			load_tile<G::KSD>(bd, tab[l].Wd, bytes_d, d_off);
			sd = tab[l].sd[dcol];
		};
		if (ug) st.embed(f, tok);
		if (ug) issue_ug(0);
		if (dn) issue_d(0);
		const bool tap = x == 0 && rank == 0 && w == 0;
		// columns rank * W + lane of the eight XCDs' partial sums of a layer's down projection
		auto sum_d = [&](int l, float &sum) -> bool {
			unsigned v[RX];
			if (!wait_near(&near_d, (unsigned)(G::CT * (l + 1)), wt)) return false;
			if (!poll_column<RX>(v, cross_view(l, G::XD, RX * H), (unsigned)(ocol + min(lane, G::W - 1)) * 4u, H * 4u, wt)) return false;
			sum = 0.0f;
#pragma unroll
			for (int i = 0; i < RX; i++) sum += __uint_as_float(v[i]);
			return true;
		};
		for (int l = 0;; l++) {
			if (l > 0) {
				if (red) {
					float sum;
					if (!sum_d(l - 1, sum)) return;
					if (lane < G::W) store_local(l - 1, G::PD + ocol + lane, sum);
					signal_near(&near_pd);
				}
				if (ug) {
					f32x4 wpo[G::NQ];
					u32x4 p[G::NQ];
					S::load(wpo, tab[l - 1].mpost);
					if (!wait_near(&near_pd, (unsigned)l, wt)) return;
					if (!poll_row<G::NQ>(p, local_view(l - 1, G::PD, H), wt)) return;
					st.add_post_norm(p, wpo);
				}
			}
			if (tap) st.store(f.xr + (size_t)(2 * l) * H);
			if (l > 0 && (ug || dn)) {  // behind the hand-over of the layer's input and its Q (see load_tile)
				if (!wait_near(&near_q, (unsigned)(l + 1), wt)) return;
				if (ug) issue_ug(l);
				if (dn) issue_d(l);
			}
			if (red) {
				if (ug) {  // ahead of its wait for the sums
					S::park(norm_s[G::UGT - 1][0], tab[l].apost);
					S::park(norm_s[G::UGT - 1][1], tab[l].mpre);
				}
				// merge of the two halves of every head's keys: weights from (maximum, sum) of the XCDs
				u32x2 ml;
				unsigned v[RX];
				const __amdgpu_buffer_rsrc_t rs = cross_view(l, 0, G::LOC);
				const unsigned c = (unsigned)(G::XO + ocol + min(lane, G::W - 1)) * 4u;
				if (!wait_near(&near_o, (unsigned)(G::CT * (l + 1)), wt)) return;
				for (int spins = 0;;) {
					ml = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, (unsigned)(lane & 7) * 128u, G::XML * 4u, AUX_DEV));
#pragma unroll
					for (int i = 0; i < RX; i++) v[i] = __builtin_amdgcn_raw_buffer_load_b32(rs, c, (unsigned)(i * H) * 4u, AUX_DEV);
					unsigned top = max(ml[0], ml[1]);
#pragma unroll
					for (int i = 0; i < RX; i++) top = max(top, v[i]);
					if (__all(top != SENTINEL)) break;
					if (!wt.again(spins)) return;
				}
				const float m = __uint_as_float(ml[0]), ls = __uint_as_float(ml[1]);
				const float M = fmaxf(m, tg_red_partner<1>(m));
				const float e = tga::attn_exp(m - M), el = __fmul_rn(e, ls);
				const float wgt = e * __builtin_amdgcn_rcpf(el + tg_red_partner<1>(el));
				float sum = 0.0f;
#pragma unroll
				for (int i = 0; i < RX; i++)
					sum = fmaf(__uint_as_float(__builtin_amdgcn_readlane((int)__float_as_uint(wgt), i)), __uint_as_float(v[i]), sum);
				if (lane < G::W) {
					store_local(l, G::PO + ocol + lane, sum);
					reset_local(l, G::PO + ocol + lane);
					reset_local(l, G::PD + ocol + lane);
				}
				signal_near(&near_po);
			}
			if (ug) {
				f32x4 wn[G::NQ];
				u32x4 p[G::NQ];
				if (!red) {
					S::park(norm_s[w][0], tab[l].apost);
					S::park(norm_s[w][1], tab[l].mpre);
				}
				if (!wait_near(&near_po, (unsigned)(l + 1), wt)) return;
				if (!poll_row<G::NQ>(p, local_view(l, G::PO, H), wt)) return;
				S::unpark(wn, norm_s[w][0]);
				st.add_post_norm(p, wn);
				S::unpark(wn, norm_s[w][1]);
				const float k = st.pre_norm_digits(wn, dg, G::PSH);
				const float y = tile_product<G::KSH>(bu, dg, G::PSH) * k * su;  // columns 0 .. 7 up, 8 .. 15 gate
				const float gate = tg_red_partner<8>(y);
				const float hv = gelu_lut(gate, lut_in_lds ? lut_s : f.lut, f.gmin, f.geps, f.lut_size) * y;
				const int at = G::HB + rank * G::PAIRS + 8 * w + lane;
				if (lane < np) {
					store_local(l, at, hv);
					reset_local(l, at);
				}
			}
			if (dn) {
				u32x4 hv[G::NQD];
				if (!poll_row<G::NQD>(hv, local_view(l, G::HB, G::KD), wt)) return;
				unsigned mb = 0;
#pragma unroll
				for (int i = 0; i < G::NQD; i++)
#pragma unroll
					for (int e = 0; e < 4; e++) mb = max(mb, hv[i][e] & 0x7fffffffu);
				float mul;
				const float inv = digit_factors(wave_max_u32(mb), mul);
#pragma unroll
				for (int i = 0; i < G::NQD; i++) {
					float u[4];
#pragma unroll
					for (int e = 0; e < 4; e++) u[e] = __uint_as_float(hv[i][e]);
					put_digits(dg, G::PSD, lane + 64 * i, u, mul);  // (rows past the slice: zeros)
				}
				const float y = tile_product<G::KSD>(bd, dg, G::PSD) * inv * sd;
				const int at = G::XD + x * H + ocol + 16 * w + lane;
				if (lane < min(16, G::W - 16 * w)) {
					store_dev(l, at, not_sentinel(y));
					store_dev(l + 2, at, SENTINEL);
				}
				signal_near(&near_d);
			}
			if (tap) st.store(f.xr + (size_t)(2 * l + 1) * H);
			if (l + 1 == f.L) break;  // (the last tiles' registers end here)
		}
		if (red) {
			float sum;
			if (!sum_d(f.L - 1, sum)) return;
			if (x == 0 && lane < G::W) f.pend[ocol + lane] = sum;
			if (lane < G::W) store_local(f.L - 1, G::PD + ocol + lane, sum);
		}
		return;
	}

	// ---- the output projection's tiles: waves 5 .. 7 ----
	const int head = x >> 1, ot = w - 5;
	const bool out = ot >= 0 && ot < G::CT;
	i32x4 bo[4];
	float so = 0.0f;
	const int ocl = out ? out_col(ot) : 0;
	const uint32_t o_off = piece_at(ocl, head * 16 + kq, 1024);
	const Keys k_local(f.pos, f.bp_local, f.n_pos_local, x, rank), k_global(f.pos, f.bp_global, f.n_pos, x, rank);
	auto keys_of = [&](int l) { return tab[l].is_sw ? k_local : k_global; };
	auto issue_o = [&](int l) {
		load_tile<4>(bo, tab[l].Wo, bytes_o, o_off);
		so = tab[l].so[ocl];
	};
	// merge of the units' attention results and the head's rows of the projection (modules.hpp:161-164)
	auto project = [&](int l, const Keys &ks) -> bool {
		const __amdgpu_buffer_rsrc_t rl = local_view(l, G::AP, 256 * ks.parts), rm = local_view(l, G::AML, 2 * RU);
		// a wait for the results' (maximum, sum), then for the results, which were stored in front of those
		constexpr int PG = 16;
		u32x2 ml;
		u32x4 pv[PG];
		const int b = lane & 31;
		const unsigned ml_at = (unsigned)min(b, ks.parts - 1) * 8u;
		auto part_at = [&](int i) { return (unsigned)min(i, ks.parts) * 1024u; };  // past the last: zeros, without a memory access
		for (int spins = 0;;) {
			ml = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rm, ml_at, 0, AUX_DEV));
			if (__all(max(ml[0], ml[1]) != SENTINEL)) break;
			if (!wt.again(spins)) return false;
		}
		for (int spins = 0;;) {
			unsigned top = 0;
#pragma unroll
			for (int i = 0; i < PG; i++) pv[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rl, (unsigned)lane * 16u, part_at(i), AUX_DEV));
#pragma unroll
			for (int i = 0; i < PG; i++) top = max(top, max4(pv[i]));
			if (__all(top != SENTINEL)) break;
			if (!wt.again(spins)) return false;
		}
		const float m = b < ks.parts ? __uint_as_float(ml[0]) : -INFINITY;
		const float M = tg_wave_max(m);
		const float e = m == -INFINITY ? 0.0f : tga::attn_exp(m - M);
		const float L = 0.5f * wave_sum(__fmul_rn(e, b < ks.parts ? __uint_as_float(ml[1]) : 0.0f));  // every part sits in two lanes
		float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
		for (int g = 0;;) {
#pragma unroll
			for (int i = 0; i < PG; i++) {
				const float ei = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(e), g + i));
#pragma unroll
				for (int c = 0; c < 4; c++) o[c] = fmaf(__uint_as_float(pv[i][c]), ei, o[c]);
			}
			g += PG;
			if (g >= ks.parts) break;
			for (int spins = 0;;) {
				unsigned top = 0;
#pragma unroll
				for (int i = 0; i < PG; i++) pv[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rl, (unsigned)lane * 16u, part_at(g + i), AUX_DEV));
#pragma unroll
				for (int i = 0; i < PG; i++) top = max(top, max4(pv[i]));
				if (__all(top != SENTINEL)) break;
				if (!wt.again(spins)) return false;
			}
		}
		unsigned mb = 0;
#pragma unroll
		for (int c = 0; c < 4; c++) mb = max(mb, __float_as_uint(o[c]) & 0x7fffffffu);
		float mul;
		const float inv = digit_factors(wave_max_u32(mb), mul);
		put_digits(dg, G::PSO, lane, o, mul);
		const float y = tile_product<4>(bo, dg, G::PSO) * inv * so;
		const int at = G::XO + x * H + ocol + 16 * ot + lane;
		if (lane < min(16, G::W - 16 * ot)) {
			store_dev(l, at, not_sentinel(y));
			store_dev(l + 2, at, SENTINEL);
		}
		signal_near(&near_o);
		if (rank == 0 && ot == 0 && lane < 2) {
			store_dev(l, G::XML + 32 * x + lane, not_sentinel(lane == 0 ? M : L));
			store_dev(l + 2, G::XML + 32 * x + lane, SENTINEL);
		}
		return true;
	};

	if (w < 6) {
		// ================ wave 4: Q tile; wave 5: K|V tile (where the token's slot is the XCD's), projection tile 0 ================
		S st;
		i32x4 bq[G::KSH];
		float sq = 0.0f;
		const int qcol = w == 4 ? head * 256 + rank * 8 + (col & 7) : 1024 + ((col & 8) ? 256 : 0) + rank * 8 + (col & 7);
		const uint32_t q_off = piece_at(qcol, kq, H);
		auto issue_qkv = [&](int l) {  // not wanted: no records, no memory access
			load_tile<G::KSH>(bq, tab[l].Wqkv, w == 4 || keys_of(l).mine ? bytes_h : 0u, q_off);
			sq = tab[l].sqkv[qcol];
		};
		const int at = G::QKV + (w == 4 ? rank * 8 + col : 256 + ((col & 8) ? 256 : 0) + rank * 8 + (col & 7));
		const bool has_col = lane < (w == 4 ? 8 : 16);
		f32x4(*nw)[64 * G::NQ] = norm_s[G::UGT + w - 4];
		st.embed(f, tok);
		issue_qkv(0);
		if (out) issue_o(0);
		for (int l = 0;; l++) {
			const Keys ks = keys_of(l);
			if (l > 0) {
				f32x4 wpo[G::NQ];
				u32x4 p[G::NQ];
				S::load(wpo, tab[l - 1].apost);
				if (!wait_near(&near_po, (unsigned)l, wt)) return;
				if (!poll_row<G::NQ>(p, local_view(l - 1, G::PO, H), wt)) return;
				st.add_post_norm(p, wpo);
				S::park(nw[0], tab[l - 1].mpost);
				S::park(nw[1], tab[l].apre);
				if (!wait_near(&near_pd, (unsigned)l, wt)) return;
				if (!poll_row<G::NQ>(p, local_view(l - 1, G::PD, H), wt)) return;
				S::unpark(wpo, nw[0]);
				st.add_post_norm(p, wpo);
			} else {
				S::park(nw[1], tab[0].apre);
			}
			if (w == 4 || ks.mine) {
				f32x4 wpre[G::NQ];
				S::unpark(wpre, nw[1]);
				const float k = st.pre_norm_digits(wpre, dg, G::PSH);
				const float y = tile_product<G::KSH>(bq, dg, G::PSH) * k * sq;
				if (has_col) store_local(l, at, y);
				if (w == 4) signal_near(&near_q);
			}
			if (has_col) reset_local(l, at);
			if (w == 4) {  // the unit's share of the attention results' slots
				*reinterpret_cast<u32x4 *>(local_of(l + 2) + G::AP + rank * 256 + 4 * lane) = u32x4{SENTINEL, SENTINEL, SENTINEL, SENTINEL};
				if (lane < 2) reset_local(l, G::AML + 2 * rank + lane);
			}
			if (out && !project(l, ks)) return;
			if (l + 1 == f.L) return;
			if (out) issue_o(l + 1);
			issue_qkv(l + 1);
		}
	}

	// ================ waves 6 and 7: attention, projection tiles 1 and 2 ================
	const int wv = w - 6;
	f32x4 kr[tga::KB], vr[tga::KB], wqn, wkn;
	auto load_rows = [&](f32x4 (&d)[tga::KB], const float *cache, int slots, int row0, bool want) {
		const uint32_t bytes = want ? (uint32_t)slots * 1024u : 0u;
		const __amdgpu_buffer_rsrc_t rc = make_rsrc(cache, bytes);
#pragma unroll
		for (int j = 0; j < tga::KB; j++) d[j] = ldx(rc, (uint32_t)lane * 16u, min((uint32_t)min(row0 + j, slots - 1) * 1024u, bytes));
	};
	auto issue_kv = [&](int l) {
		const Keys ks = keys_of(l);
		const int row0 = ks.first + 8 * (AW * max(ks.part, 0) + wv);
		const bool want = ks.part >= 0 && row0 < ks.first + ks.n;
		load_rows(kr, tab[l].kc, ks.max_pos, row0, want);
		load_rows(vr, tab[l].vc, ks.max_pos, row0, want);
		wqn = *reinterpret_cast<const f32x4 *>(tab[l].rms_q + 4 * lane);
		wkn = *reinterpret_cast<const f32x4 *>(tab[l].rms_k + 4 * lane);
	};
	issue_kv(0);
	if (out) issue_o(0);
	// this position's rotations, of global and local layers: dims 4 lane .. of each half
	const size_t rot = (size_t)f.pos * 128 + 4 * (lane & 31);
	const f32x4 cg = *reinterpret_cast<const f32x4 *>(f.cos_g + rot), sg = *reinterpret_cast<const f32x4 *>(f.sin_g + rot);
	const f32x4 cl = *reinterpret_cast<const f32x4 *>(f.cos_l + rot), sl = *reinterpret_cast<const f32x4 *>(f.sin_l + rot);

	for (int l = 0;; l++) {
		const Keys ks = keys_of(l);
		const bool sw = tab[l].is_sw != 0;
		const f32x4 c4 = sw ? cl : cg, s4 = sw ? sl : sg;
		u32x4 qv[3];
		// the token's own key and value only where they are computed; a unit without keys waits as well: it may not run ahead
		// of the ring
		if (!wait_near(&near_q, (unsigned)(l + 1), wt)) return;
		if (!poll_row<3>(qv, local_view(l, G::QKV, ks.mine ? 768 : 256), wt)) return;
		if (ks.part >= 0) {
			const f32x4 q = __builtin_bit_cast(f32x4, tga::attn_head_finish(__builtin_bit_cast(tga::af4, qv[0]), __builtin_bit_cast(tga::af4, wqn),
			                                                               __builtin_bit_cast(tga::af4, c4), __builtin_bit_cast(tga::af4, s4), 0.0625f));  // ops.hpp:257
			// (not the own token's XCD: key and value read as zeros, and no slot is taken for theirs)
			const f32x4 knew = __builtin_bit_cast(f32x4, tga::attn_head_finish(__builtin_bit_cast(tga::af4, qv[1]), __builtin_bit_cast(tga::af4, wkn),
			                                                                  __builtin_bit_cast(tga::af4, c4), __builtin_bit_cast(tga::af4, s4), 1.0f));
			const f32x4 vnew = __builtin_bit_cast(f32x4, qv[2]);
			float m_run = -INFINITY, l_run = 0.0f;
			f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
			const int blocks = (ks.n + 7) >> 3, stride = AW * ks.parts;
			const int jl = lane >> 3;  // the key whose score this lane ends up with
			for (int t = AW * ks.part + wv; t < blocks; t += stride) {
				const int row0 = ks.first + 8 * t;
				if (t != AW * ks.part + wv) {
					load_rows(kr, tab[l].kc, ks.max_pos, row0, true);
					load_rows(vr, tab[l].vc, ks.max_pos, row0, true);
				}
				float d[tga::KB];
#pragma unroll
				for (int j = 0; j < tga::KB; j++) {
					const f32x4 kv = (row0 + j == ks.cur) ? knew : kr[j];
					d[j] = fmaf(q[3], kv[3], fmaf(q[2], kv[2], fmaf(q[1], kv[1], q[0] * kv[0])));
				}
				// summed over the lanes and dealt out: keys 4 .. 7 stay with the upper half, odd pairs with odd rows, odd keys
				// with the upper eight lanes of a row
#pragma unroll
				for (int j = 0; j < 4; j++) {
					const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(d[j]), __float_as_uint(d[j + 4]), false, false);
					d[j] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
				}
#pragma unroll
				for (int j = 0; j < 2; j++) {
					const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(d[j]), __float_as_uint(d[j + 2]), false, false);
					d[j] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
				}
				const bool b3 = (lane & 8) != 0;
				const float keep = b3 ? d[1] : d[0], send = b3 ? d[0] : d[1];
				float s = keep + tga::attn_dpp<0x128>(send);  // row_ror:8
				s += tga::attn_dpp<0x141>(s);                 // row_half_mirror
				s += tga::attn_dpp<0x1B>(s);                  // quad_perm:[3,2,1,0]
				s += tga::attn_dpp<0xB1>(s);                  // quad_perm:[1,0,3,2]
				const bool ok = 8 * t + jl < ks.n;
				s = ok ? s : -INFINITY;
				const float m_new = fmaxf(m_run, tg_wave_max(s));  // the first key of a block is always valid
				const float p = ok ? tga::attn_exp(s - m_new) : 0.0f;
				const float scale = tga::attn_exp(m_run - m_new);
				l_run = fmaf(l_run, scale, 0.125f * wave_sum(p));  // every weight sits in eight lanes
				m_run = m_new;
				acc *= scale;
#pragma unroll
				for (int j = 0; j < tga::KB; j++) {
					const f32x4 vv = (row0 + j == ks.cur) ? vnew : vr[j];
					const float pj = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(p), 8 * j));
#pragma unroll
					for (int e = 0; e < 4; e++) acc[e] = fmaf(pj, vv[e], acc[e]);
				}
				if (head == 0 && ks.mine && ks.cur >= row0 && ks.cur < row0 + 8) {  // KVCache::update_single, decode.hpp:49-70
					*reinterpret_cast<f32x4 *>(tab[l].kc + (size_t)ks.cur * 256 + 4 * lane) = knew;
					*reinterpret_cast<f32x4 *>(tab[l].vc + (size_t)ks.cur * 256 + 4 * lane) = vnew;
				}
			}
			// the two waves' results meet in LDS; the one that arrives last merges them
			*reinterpret_cast<f32x4 *>(&pacc[wv][4 * lane]) = acc;
			if (lane == 0) {
				pm[wv] = m_run;
				pl[wv] = l_run;
			}
			unsigned old = 0;
			if (lane == 0) old = __hip_atomic_fetch_add(&arrived, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
			old = (unsigned)__builtin_amdgcn_readfirstlane((int)old);
			if (old & 1u) {
				const float m0 = pm[0], m1 = pm[1], M = fmaxf(m0, m1);  // (a wave without keys: -inf, and both may be)
				const float e0 = m0 == -INFINITY ? 0.0f : tga::attn_exp(m0 - M), e1 = m1 == -INFINITY ? 0.0f : tga::attn_exp(m1 - M);
				const f32x4 a0 = *reinterpret_cast<const f32x4 *>(&pacc[0][4 * lane]), a1 = *reinterpret_cast<const f32x4 *>(&pacc[1][4 * lane]);
				u32x4 ov;
#pragma unroll
				for (int c = 0; c < 4; c++) ov[c] = not_sentinel(fmaf(a1[c], e1, __fmul_rn(a0[c], e0)));  // the same sum whoever merges
				const float ls = fmaf(pl[1], e1, __fmul_rn(pl[0], e0));
				*reinterpret_cast<u32x4 *>(local_of(l) + G::AP + ks.part * 256 + 4 * lane) = ov;
				if (lane == 0) *reinterpret_cast<u32x2 *>(local_of(l) + G::AML + 2 * ks.part) = u32x2{not_sentinel(M), not_sentinel(ls)};
			}
		}
		if (out && !project(l, ks)) return;
		if (l + 1 == f.L) return;
		issue_kv(l + 1);
		if (out) issue_o(l + 1);
	}
}

__global__ void deal_kernel(int *out) {
	int xcc;
	asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(xcc));
	if (threadIdx.x == 0) out[blockIdx.x] = xcc;
}

}  // namespace

// The launch counts on 32 workgroups on each of eight XCDs, workgroup b being the (b / 8)th of its own.
bool tg_resident_device(int n_cu, hipStream_t s) {
	if (n_cu != RX * RU) return false;
	int *d = nullptr, h[RX * RU];
	if (hipMalloc((void **)&d, sizeof(h)) != hipSuccess) return false;
	hipLaunchKernelGGL(deal_kernel, dim3(RX * RU), dim3(RNT), 0, s, d);
	bool ok = hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, s) == hipSuccess && hipStreamSynchronize(s) == hipSuccess;
	(void)hipFree(d);
	for (int g = 0; ok && g < RU; g++) {
		unsigned seen = 0;
		for (int i = 0; i < RX; i++) seen |= 1u << (h[RX * g + i] & 31);
		ok = seen == (1u << RX) - 1u;
	}
	return ok;
}

bool tg_resident_shape(int hidden, int ff) { return (hidden == 640 && ff == 2048) || (hidden == 1152 && ff == 6912); }

size_t tg_resident_exchange_words(int hidden) { return 4 * (size_t)(hidden == 640 ? Geo<640, 2048>::SLOT : Geo<1152, 6912>::SLOT); }

void tg_launch_decode_resident(const TgResident &f, int hidden, hipStream_t s) {
	const dim3 grid(RX * RU), block(RNT);
	if (hidden == 640) hipLaunchKernelGGL((decode_resident_kernel<640, 2048>), grid, block, 0, s, f);
	else hipLaunchKernelGGL((decode_resident_kernel<1152, 6912>), grid, block, 0, s, f);
}
