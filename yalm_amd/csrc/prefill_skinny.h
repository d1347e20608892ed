// prefill_skinny.h — the prefill's GEMMs for a SHORT prompt (T <= 64 rows: the
// CLI's prompt hydration, main.cpp:91-97 in the reference, runs T one-token
// forwards there), and the sums of K slices. At small T the 256-row tiles of
// prefill_gemm.h leave most CUs idle (Llama-3B Wo / W2, N 3072: 12-16 tiles) and the
// GEMM is a weight stream, not MFMA work: every weight byte is read once, for T <= 64 rows.
//
//   stream_gemm_kernel: a workgroup owns 16 weight rows per wave and a slice of K; weight
//     rows and A rows (tokens) come through one ring of LDS-DMA stages; the TOKENS are the
//     MFMA's A operand, the weight rows B. One slice: the epilogue runs in the launch;
//     several: each leaves f32 partials part[ks][row][col].
//   skinny_reduce_kernel: per (16 rows x 16 FJ columns) wave block, the KS partials
//     summed in ks order (deterministic) into the 16x16 MFMA C layout, then the same
//     epilogue object as the large-tile GEMM (prefill_gemm.h E16*: RoPE + cache
//     write, residual add, GLU).
//   reduce_norm_rows_kernel: the same for a residual product, with the next row norm.
#pragma once

#include "prefill_gemm.h"

namespace pf {

// C = A · W^T for T <= 16 MT rows. Workgroup = NW waves x 16 weight rows, stages of 128 K columns
// (ROWB bytes per weight row) in a ring of NS: per stage a wave DMAs its own 16 weight rows and its
// share of the A rows, all waves read A. One barrier per stage publishes the stage that landed and
// frees the slot of the one before it, which the next DMA refills.
//
// What bounds it is the weight stream: 16 NW ROWB bytes a stage with NS - 1 stages in flight, two
// workgroups per CU where the ring fits 80 KB (64-96 KB in flight per CU: HBM latency x bandwidth is about
// 55 KB per CU), else one. A slice may be the whole of K: a gated pair of 448 row blocks is one round of
// workgroups that never refill their pipeline, and its epilogue needs no partials. (The form before it
// staged a whole A chunk per workgroup and so cut K into chunks of at most 32 KB of A: at 13 rows, W1 | W3 of
// Mistral-7B was 1792 workgroups, 52.4 + 4.7 us for 235 MB.)
//
// DUAL: columns >= c_split take A = [hi | lo], kb columns apart, against the same weights (the split-f16
// K / V operand): the weight fragment is read once for both halves.
//
// 16-byte chunks are XOR-swizzled on the source side of the DMA so that 16 rows' fragment reads of one
// chunk column spread over the banks: A (256-byte rows) by row & 15, f16 weights the same, E5M2 (128-byte
// rows, two per 256 bytes) by (row >> 1) & 7.
template <int MT, int NW, class BMAP, bool DUAL>
struct StreamCfg {
	static constexpr int EB = sizeof(bmap_elt<BMAP>);
	static constexpr int KSTG = 128, ROWB = KSTG * EB;
	static constexpr int WB = NW * 16 * ROWB, AB = 16 * MT * KSTG * 2; // stage bytes: weights, one half of A
	static constexpr int SB = WB + AB * (DUAL ? 2 : 1);
	static constexpr int FIT2 = 81920 / SB, FIT1 = 163840 / SB;
	static constexpr int NS = FIT2 >= 3 ? (FIT2 < 6 ? FIT2 : 6) : (FIT1 < 4 ? FIT1 : 4);
	static constexpr int NWI = ROWB / 64;          // weight DMAs per wave and stage: 16 ROWB bytes, 1 KB each
	static constexpr int NA = 4 * MT / NW;         // A DMAs per wave, stage and half
	static constexpr size_t RED = (size_t)NW * MT * 16 * 17 * 4; // the epilogue's sums
	static constexpr size_t LDS = (size_t)NS * SB > RED ? (size_t)NS * SB : RED;
	static_assert(NA * NW == 4 * MT && NS >= 2, "shape");
};
struct NoEpi {}; // partials

template <int MT, int NW, class BMAP, bool DUAL, bool GLU, class EPI, bool BF>
__global__ __launch_bounds__(64 * NW) void stream_gemm_kernel(const uint16_t *__restrict__ A, int lda, int T, int nst_all,
                                                              int kb, BMAP bm, int nblk, int nsc, int c_split, int Np,
                                                              float *__restrict__ part, EPI epi, int drain) {
	using C = StreamCfg<MT, NW, BMAP, DUAL>;
	using elt = bmap_elt<BMAP>;
	constexpr int EB = C::EB, NS = C::NS, CW = C::NWI + C::NA;
	extern __shared__ __attribute__((aligned(16))) char smem_c[];
	const int nb = blockIdx.x % nblk, ks = blockIdx.x / nblk;
	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int n = lane & 15, q = lane >> 4;
	const int cb = nb * 16 * NW;        // the workgroup's first B row (output column)
	const bool dual = DUAL && cb >= c_split;
	const int st0 = ks * nsc, nst = min(nsc, nst_all - st0);
	const int k0 = st0 * C::KSTG;
	const elt *wsrc[C::NWI];
#pragma unroll
	for (int i = 0; i < C::NWI; ++i) {
		const int rr = EB == 2 ? 4 * i + (lane >> 4) : 8 * i + (lane >> 3);
		const int ch = EB == 2 ? (lane & 15) ^ rr : (lane & 7) ^ ((rr >> 1) & 7);
		wsrc[i] = bm.row(cb / BMAP::COLS_PER_TILE_DIV, 16 * wave + rr, kb) + k0 + 16 / EB * ch;
	}
	const uint16_t *asrc[C::NA];
#pragma unroll
	for (int i = 0; i < C::NA; ++i) { // rows past T repeat the last one (their results are dropped)
		const int r = 4 * (wave * C::NA + i) + (lane >> 4);
		asrc[i] = A + (size_t)min(r, T - 1) * lda + k0 + 8 * ((lane & 15) ^ (r & 15));
	}
	// the workgroups walk the slice's columns from different stages on: rows are a power of two apart, so
	// workgroups in step would all read the same HBM channels
	const int rot = nb % nst;
	auto issue = [&](int st) {
		char *const base = smem_c + (st % NS) * C::SB;
		st = st + rot < nst ? st + rot : st + rot - nst;
#pragma unroll
		for (int i = 0; i < C::NWI; ++i)
			__builtin_amdgcn_global_load_lds((const void *)(wsrc[i] + st * C::KSTG),
			                                 (YALM_LDS void *)(base + (wave * C::NWI + i) * 1024), 16, 0, 0);
#pragma unroll
		for (int i = 0; i < C::NA; ++i)
			__builtin_amdgcn_global_load_lds((const void *)(asrc[i] + st * C::KSTG),
			                                 (YALM_LDS void *)(base + C::WB + (wave * C::NA + i) * 1024), 16, 0, 0);
		if (DUAL && dual)
#pragma unroll
			for (int i = 0; i < C::NA; ++i)
				__builtin_amdgcn_global_load_lds((const void *)(asrc[i] + kb + st * C::KSTG),
				                                 (YALM_LDS void *)(base + C::WB + C::AB + (wave * C::NA + i) * 1024), 16, 0, 0);
	};
	for (int st = 0; st < min(NS - 1, nst); ++st)
		issue(st);
	f32x4_t acc[MT];
#pragma unroll
	for (int m = 0; m < MT; ++m)
		acc[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
	for (int st = 0; st < nst; ++st) {
		// stage st has landed: the NS - 2 stages after it stay in flight (near the slice's end: drain)
		if (st + NS - 2 >= nst || drain)
			asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
		else if (DUAL && dual)
			asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * (CW + C::NA)) : "memory");
		else
			asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * CW) : "memory");
		raw_barrier(); // ... every wave's share of it, and everyone is done reading stage st - 1
		if (st + NS - 1 < nst)
			issue(st + NS - 1);
		const char *const base = smem_c + (st % NS) * C::SB;
		const char *const bst = base + wave * 16 * C::ROWB + n * C::ROWB;
		const uint16_t *const as = (const uint16_t *)(base + C::WB);
#pragma unroll
		for (int j = 0; j < 4; ++j) {
			half8_t b;
			if constexpr (EB == 2)
				b = *(const half8_t *)(bst + 16 * ((4 * j + q) ^ n));
			else // E5M2: 8 of a chunk's 16 columns
				b = e5m2x8(*(const uint2 *)(bst + 16 * ((2 * j + (q >> 1)) ^ ((n >> 1) & 7)) + 8 * (q & 1)));
#pragma unroll
			for (int m = 0; m < MT; ++m) {
				const uint16_t *const ap = as + (16 * m + n) * C::KSTG + 8 * ((4 * j + q) ^ n);
				acc[m] = mfma16<BF>(*(const half8_t *)ap, b, acc[m]);
				if (DUAL && dual)
					acc[m] = mfma16<BF>(*(const half8_t *)(ap + C::AB / 2), b, acc[m]);
			}
		}
	}
	if constexpr (std::is_same<EPI, NoEpi>::value) {
		float *pp = part + (size_t)ks * 16 * MT * Np + cb + 16 * wave + n;
#pragma unroll
		for (int m = 0; m < MT; ++m)
#pragma unroll
			for (int r = 0; r < 4; ++r)
				pp[(size_t)(16 * m + crow16(r, lane)) * Np] = acc[m][r];
	} else {
		// the waves' columns meet in LDS: a wave then runs the epilogue of one 16-row tile x 64 columns
		raw_barrier();
		float *const red = (float *)smem_c;
#pragma unroll
		for (int m = 0; m < MT; ++m)
#pragma unroll
			for (int r = 0; r < 4; ++r)
				red[((wave * MT + m) * 16 + crow16(r, lane)) * 17 + n] = acc[m][r];
		raw_barrier();
		for (int task = wave; task < MT * (NW / 4); task += NW) {
			const int m = task % MT, g = task / MT;
			if (16 * m >= T)
				continue;
			f32x4_t a2[1][4];
#pragma unroll
			for (int j = 0; j < 4; ++j)
#pragma unroll
				for (int r = 0; r < 4; ++r)
					a2[0][j][r] = red[(((4 * g + j) * MT + m) * 16 + crow16(r, lane)) * 17 + n];
			epi.template apply<1, 4>(a2, 16 * m, GLU ? cb / 2 + 32 * g : cb + 64 * g, lane, 0, 1);
		}
	}
}

// One wave per (16 rows, 16 FJ columns) block of C: the KS partials summed
// in ks order, then epi.apply<1, FJ>(acc, row0, n0, ...) exactly as the large-tile GEMM's
// epilogue sees its fragments. n0: the block's first output column, or (GLU) its first
// hidden column (BRowsGlu: 16 FJ B rows = 8 FJ W1 rows then the same 8 FJ W3 rows).
// Columns < c_split sum KS partial slots, the others KS2 (the QKV buffer: the k | v
// GEMM ran 2 KS K chunks).
template <int FJ, bool GLU, class EPI>
__global__ __launch_bounds__(256) void skinny_reduce_kernel(const float *__restrict__ part, int KS, int KS2,
                                                            int c_split, int TP, int T, int N, EPI epi) {
	const int lane = threadIdx.x & 63;
	const int gw = blockIdx.x * 4 + (threadIdx.x >> 6); // global wave = block (row tile, col block)
	const int ncb = N / (16 * FJ);
	const int rt = gw / ncb, cb = gw % ncb;
	if (rt * 16 >= T)
		return;
	const int nks = cb * 16 * FJ < c_split ? KS : KS2;
	// the KS partials of this lane's 4 FJ values: all 4 FJ loads of 4 consecutive ks in
	// flight at once, summed in ks order (deterministic; round 4's first cut ran one serial
	// chain of KS dependent loads per value: 27 us per Wo / W2 reduce at T = 1)
	f32x4_t acc[1][FJ];
	size_t off[FJ][4];
#pragma unroll
	for (int j = 0; j < FJ; ++j) {
		acc[0][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
		for (int r = 0; r < 4; ++r)
			off[j][r] = (size_t)(16 * rt + crow16(r, lane)) * N + cb * 16 * FJ + 16 * j + (lane & 15);
	}
	const size_t kstride = (size_t)TP * N;
	int ks = 0;
	for (; ks + 4 <= nks; ks += 4) {
		float v[4][FJ][4];
#pragma unroll
		for (int q = 0; q < 4; ++q)
#pragma unroll
			for (int j = 0; j < FJ; ++j)
#pragma unroll
				for (int r = 0; r < 4; ++r)
					v[q][j][r] = part[(size_t)(ks + q) * kstride + off[j][r]];
#pragma unroll
		for (int q = 0; q < 4; ++q)
#pragma unroll
			for (int j = 0; j < FJ; ++j)
#pragma unroll
				for (int r = 0; r < 4; ++r)
					acc[0][j][r] += v[q][j][r];
	}
	for (; ks < nks; ++ks) {
#pragma unroll
		for (int j = 0; j < FJ; ++j)
#pragma unroll
			for (int r = 0; r < 4; ++r)
				acc[0][j][r] += part[(size_t)ks * kstride + off[j][r]];
	}
	const int n0 = GLU ? cb * 8 * FJ : cb * 16 * FJ;
	epi.template apply<1, FJ>(acc, 16 * rt, n0, lane, 0, 1);
}

// The partials of a residual product (Wo, W2), the residual add and the NEXT row norm in one launch:
// row t's KS slots summed in slot order, X[t] += scale * sum (E16Residual's arithmetic), then Xn[t] =
// f16(rmsnorm(X[t]) * w) (rmsnorm_rows_kernel's; SPLIT: [hi | lo]). One workgroup per row holds the row in
// registers (NV float4 per thread), so the row is neither written and read again between the two nor
// waited for by a second launch. What bounds it at few rows is the chain load - sum - barrier - store, not
// bytes. Measured (Mistral-7B, 13 rows): 5.3 us reduce + 10.4 us norm before. w null: the residual add alone.
template <bool SPLIT, int NV>
__global__ void reduce_norm_rows_kernel(const float *__restrict__ part, int KS, size_t kstride, float *__restrict__ X,
                                        int dim, float scale, const float *__restrict__ w, float eps,
                                        uint16_t *__restrict__ Xn, unsigned *range) {
	__shared__ float red[16];
	const int t = blockIdx.x, nt = blockDim.x, tid = threadIdx.x;
	float *x = X + (size_t)t * dim;
	const float *p = part + (size_t)t * dim;
	// every index clamped into the row, the sums and stores of the lanes past it left out: the
	// loads stay unconditional, all NV of them (and KB slots of each) in flight together
	int at[NV];
	float4_t v[NV], g[NV], acc[NV];
#pragma unroll
	for (int k = 0; k < NV; ++k) {
		at[k] = min(4 * (tid + nt * k), dim - 4);
		v[k] = *(const float4_t *)(x + at[k]);
		g[k] = w ? *(const float4_t *)(w + at[k]) : float4_t{0.f, 0.f, 0.f, 0.f};
		acc[k] = float4_t{0.f, 0.f, 0.f, 0.f};
	}
	constexpr int KB = NV == 1 ? 8 : 4;
	for (int k0 = 0; k0 < KS; k0 += KB) {
		float4_t b[KB][NV];
#pragma unroll
		for (int q = 0; q < KB; ++q)
#pragma unroll
			for (int k = 0; k < NV; ++k)
				b[q][k] = *(const float4_t *)(p + (size_t)min(k0 + q, KS - 1) * kstride + at[k]);
#pragma unroll
		for (int q = 0; q < KB; ++q)
			if (k0 + q < KS)
#pragma unroll
				for (int k = 0; k < NV; ++k)
					acc[k] += b[q][k];
	}
	float ss = 0.0f;
#pragma unroll
	for (int k = 0; k < NV; ++k) {
		const bool in = 4 * (tid + nt * k) < dim;
#pragma unroll
		for (int e = 0; e < 4; ++e)
			v[k][e] += acc[k][e] * scale;
		if (in) {
			*(float4_t *)(x + at[k]) = v[k];
			ss += v[k][0] * v[k][0] + v[k][1] * v[k][1] + v[k][2] * v[k][2] + v[k][3] * v[k][3];
		}
	}
	if (!w)
		return;
	ss = wave_sum(ss);
	if ((tid & 63) == 0)
		red[tid >> 6] = ss;
	__syncthreads();
	float tot = 0.0f;
	for (int i = 0; i < (nt + 63) >> 6; ++i)
		tot += red[i];
	const float rs = 1.0f / sqrtf(tot / dim + eps);
	uint16_t *row = Xn + (size_t)t * dim * (SPLIT ? 2 : 1);
	float ymax = 0.0f;
#pragma unroll
	for (int k = 0; k < NV; ++k) {
		if (4 * (tid + nt * k) >= dim)
			continue;
		float y[4];
		uint16_t hb[4];
#pragma unroll
		for (int e = 0; e < 4; ++e) {
			y[e] = v[k][e] * rs * g[k][e];
			hb[e] = f2h_bits(y[e]);
			ymax = fmaxf(ymax, y[e] != y[e] ? __builtin_inff() : fabsf(y[e])); // NaN counts as inf
		}
		*(uint2 *)(row + at[k]) = make_uint2(hb[0] | ((uint32_t)hb[1] << 16), hb[2] | ((uint32_t)hb[3] << 16));
		if constexpr (SPLIT) {
			uint16_t lb[4];
#pragma unroll
			for (int e = 0; e < 4; ++e)
				lb[e] = f2h_bits(y[e] - h2f(hb[e]));
			*(uint2 *)(row + dim + at[k]) = make_uint2(lb[0] | ((uint32_t)lb[1] << 16), lb[2] | ((uint32_t)lb[3] << 16));
		}
	}
	range_note(range, ymax, ymax);
}

} // namespace pf
