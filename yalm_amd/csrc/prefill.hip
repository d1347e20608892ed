// prefill.hip — C ABI of the batched prefill / perplexity path (prefill.h):
// yalm_prefill (prompt hydration + per-position log p(next), replacing the
// reference's position-by-position loop in main.cpp:128-200 / 91-97) and
// its kernel-level test hooks (yalm_gemm_f16, yalm_attn_prefill).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "decoder.h"
#include "prefill.h"
#include "prefill_gemm.h"
#include "prefill_skinny.h"

// Large-tile GEMM form per GEMM kind (prefill_gemm.h): the tile width BN of the
// 256-row tile. Default: auto -- the BN dividing N that minimises rounds x (BN + 64),
// rounds = ceil(tiles / CUs): a 256-CU chip should get whole rounds of large tiles
// (Llama-3B Wo / W2 N 3072 -> 192). Other exact forms (the tests, ablations) are chosen
// explicitly through yalm_set_prefill_forms: "qkv:256,wo:128,..." forces widths, 8p:0
// the 2-phase kernel, persist:0 one workgroup per tile, skinny:0 the large tiles at
// T <= 64 too (prefill_skinny.h otherwise), qkv1:0 the q and k | v GEMMs as two
// launches, skl:0 the streamed short-prompt GEMMs with every stage drained,
// ksplit:0 no K slices (plan_split), wnorm:0 the workgroup-per-row norm kernel instead of one wave per row.
// The production library reads no environment for them; the A/B build (-DYALM_AB)
// takes a decoder's initial forms from YALM_PF_FORMS (same syntax).
static int parse_pf_forms(const char *spec, PfForms &f) {
	static const char *names[6] = {"qkv", "wo", "glu", "w2", "cls", "test"};
	f = PfForms{};
	if (!spec)
		return YALM_OK;
	const char *p = spec;
	while (*p) {
		char key[16];
		int val = 0, n = 0;
		if (sscanf(p, "%15[^:,]:%d%n", key, &val, &n) != 2) {
			set_err(std::string("yalm_set_prefill_forms: bad spec at '") + p + "'");
			return YALM_ERR_ARG;
		}
		bool known = false;
		for (int k = 0; k < 6; ++k)
			if (!strcmp(key, names[k])) {
				ARGCHK(val == 128 || val == 192 || val == 256 || val == 320,
				       "yalm_set_prefill_forms: a tile width is 128, 192, 256 or 320");
				f.g16[k] = val;
				known = true;
			}
		if (!strcmp(key, "8p"))
			f.p8 = val != 0, known = true;
		else if (!strcmp(key, "persist"))
			f.persist = val != 0, known = true;
		else if (!strcmp(key, "skinny"))
			f.no_skinny = val == 0, known = true;
		else if (!strcmp(key, "qkv1"))
			f.qkv1 = val != 0, known = true;
		else if (!strcmp(key, "skl"))
			f.skl = val != 0, known = true;
		else if (!strcmp(key, "split"))
			f.split = val != 0, known = true;
		else if (!strcmp(key, "ksplit"))
			f.ksplit = val != 0, known = true;
		else if (!strcmp(key, "wnorm"))
			f.wnorm = val != 0, known = true;
		if (!known) {
			set_err(std::string("yalm_set_prefill_forms: unknown key '") + key + "'");
			return YALM_ERR_ARG;
		}
		p += n;
		if (*p == ',')
			++p;
	}
	return YALM_OK;
}

PfForms pf_forms_default() {
	PfForms f;
	if (parse_pf_forms(ab_env("YALM_PF_FORMS"), f) != YALM_OK)
		f = PfForms{};
	return f;
}

static PfForms g_test_forms; // the forms of the yalm_gemm_f16 test hook

extern "C" int yalm_set_prefill_precision(yalm_decoder d, int mode) {
	ARGCHK(d && (mode == YALM_PREFILL_FAST || mode == YALM_PREFILL_SPLIT), "yalm_set_prefill_precision: bad argument");
	d->pf_forms.split = mode == YALM_PREFILL_SPLIT;
	return YALM_OK;
}

extern "C" int yalm_set_prefill_forms(yalm_decoder d, const char *spec) {
	PfForms f;
	TRY(parse_pf_forms(spec, f));
	if (d)
		d->pf_forms = f;
	else
		g_test_forms = f;
	return YALM_OK;
}

namespace {

enum { PG_QKV = 0, PG_WO = 1, PG_GLU = 2, PG_W2 = 3, PG_CLS = 4, PG_TEST = 5 };
// range-guard slots per layer (PrefillBufs::range), in the order the pass produces them;
// the final norm's operand is slot RG_XATT of row n_layers
enum { RG_XATT = 0, RG_Q = 1, RG_XFFN = 2, RG_H = 3, RG_N = 4 };

int pf_alloc(yalm_decoder_s *d, void **p, size_t bytes) {
	HIPCHK(hipMalloc(p, bytes ? bytes : 4));
	d->dev_allocs.push_back(*p);
	return YALM_OK;
}

// BN for a GEMM of M x N (n_eff = B rows: 2 x hidden for the GLU); 0 = none fits. A
// forced width that does not divide N falls back to the automatic choice. ragged: no width needs to
// divide N (BRowsRagged), the last tile counts whole.
// e5m2: the widths of the 8-phase kernel alone (it reads the bytes as they are).
int pick_bn(const PfForms &f, int kind, int M, int n_eff, bool glu, bool ragged = false, bool e5m2 = false) {
	static const int cands[4] = {128, 192, 256, 320};
	auto fits = [&](int bn) { return (!e5m2 || (bn <= 256 && (!glu || bn == 256))) && (n_eff % bn == 0 || (ragged && bn <= 256)) && (!glu || bn == 128 || bn == 256); };
	const int form = f.g16[kind];
	if (form > 0 && fits(form) && (form == 128 || form == 192 || form == 256 || form == 320))
		return form;
	const long ncu = device_cu_count();
	const long tiles_m = (M + pf::G_BM - 1) / pf::G_BM;
	int best = 0;
	long best_cost = 0;
	for (int bn : cands) {
		if (!fits(bn))
			continue;
		const long rounds = (tiles_m * ((n_eff + bn - 1) / bn) + ncu - 1) / ncu;
		// an 8-phase tile (widths 192, 256) costs 3/4 of a 2-phase tile of the same
		// width (Llama-3B T 4096, one process: Wo / W2 at 256 in the 8-phase kernel beat
		// 192 in the 2-phase one, profiles/r3_prefill_8phase.txt)
		const long cost = rounds * (bn + 64) * (f.p8 && (bn == 192 || bn == 256) ? 3 : 4);
		if (!best || cost < best_cost || (cost == best_cost && bn > best)) {
			best = bn;
			best_cost = cost;
		}
	}
	return best;
}

// A GEMM of few rows on the large tiles: tile width bn, K in slices of nkc K tiles (ks of them; ks2 of
// the deeper columns). ks = 1: not split.
struct SplitPlan {
	int bn = 0, nkc = 1 << 24, ks = 1, ks2 = 1, n = 0;
};
int slices(int K, int nkc) { return (K / pf::BK + nkc - 1) / nkc; }

// Time of one round of 256-row tiles, in us per K tile of 64 and per tile (pipeline fill, epilogue), as
// measured with the chip full (Mistral-7B: 391 rows, W1 | W3, 64 K tiles at width 256, 93-100 us; the 104
// K tiles of its QKV, Wo and W2 slices at width 128, 129 us; 1001 rows, QKV slices of 32 at 256, 58 us), and
// a slot's f32 traffic (written, and read back from L2 and the Infinity Cache at about 5 TB/s: 45 MB in the
// 10 us of a 391-row reduce + norm). The whole is the rounds that the busiest CU walks; the deeper columns
// (Nd of depth Kd) count by their own slices. Split only where that model gains a tenth: the partials are
// extra bytes. Mistral-7B, 391 rows, QKV + Wo + W2 of a layer: 425 us whole, 129 us + 28 us of sums in slices.
// (a whole tile's epilogue, with its bias, activation or rotation, costs more than a slice's plain stores)
constexpr float T8P_KT[3] = {1.05f, 1.3f, 1.55f}, T8P_TILE = 5.0f, T8P_EPI = 4.0f; // widths 128, 192, 256
// ragged: the last tile may reach past N (n: the columns as whole tiles).
SplitPlan plan_split(const PfForms &f, int kind, int M, int Nt, int K, int Nd, int Kd, bool glu, size_t cap,
                     bool ragged = false) {
	SplitPlan best;
	if (!f.ksplit || !f.p8 || f.g16[kind] > 0)
		return best;
	const long ncu = device_cu_count(), tm = (M + pf::G_BM - 1) / pf::G_BM, TP = (M + 15) / 16 * 16;
	const int nk = K / pf::BK, nkd = Nd ? Kd / pf::BK : 0;
	float whole = 0.0f, least = 0.0f;
	for (int w = 0; w < 3; ++w) {
		const int bn = 128 + 64 * w, N = ragged ? (Nt + bn - 1) / bn * bn : Nt;
		if (N % bn || Nd % bn || (glu && bn != 256))
			continue;
		for (int ks = 1; ks <= 16; ++ks) {
			const int nkc = (nk + ks - 1) / ks;
			if (ks > 1 && (nkc < 4 || nkc == (nk + ks - 2) / (ks - 1)))
				continue;
			const int k1 = (nk + nkc - 1) / nkc, k2 = Nd ? (nkd + nkc - 1) / nkc : 1;
			if (ks > 1 && (size_t)std::max(k1, k2) * TP * (N + Nd) > cap)
				break;
			// (not split, two depths: the deep tiles alone, or the mean over the CUs)
			const long items = tm * (N / bn * k1 + Nd / bn * k2);
			float t = (float)((items + ncu - 1) / ncu) * (nkc * T8P_KT[w] + T8P_TILE + (ks == 1 ? T8P_EPI : 0.0f));
			if (ks == 1 && Nd)
				t = std::max((float)nkd, (float)(tm * (N / bn * nk + Nd / bn * nkd)) / ncu) * T8P_KT[w] + T8P_TILE + T8P_EPI;
			if (ks == 1) {
				whole = whole == 0.0f ? t : std::min(whole, t);
				continue;
			}
			t += 3.0f + (float)((long)k1 * N + (long)k2 * Nd) * M * 8.0f / 5e6f;
			if (least == 0.0f || t < least) {
				least = t;
				best = {bn, nkc, k1, k2, N};
			}
		}
	}
	return best.ks > 1 && least < 0.9f * whole ? best : SplitPlan{};
}

template <class EPI, class BMAP, int FJ0, int FJ1>
int launch_g8p(const PfForms &f, const uint16_t *A, int lda, int M, int K, int kb, const BMAP &bm, int N,
               const EPI &epi, hipStream_t st, int c0, int c_split = -1, int K2 = 0, int nkc = 1 << 24);

// The K slices' partials of C = A B^T into `part` ([slot][16-row-rounded M][N + Nd]); columns [N, N + Nd)
// (Nd > 0: width 256) run depth Kd
template <class BMAP, bool BF = false>
int launch_split(const PfForms &f, const SplitPlan &s, const uint16_t *A, int lda, int M, int K, int kb, const BMAP &bm,
                 int N, int Nd, int Kd, float *part, hipStream_t st) {
	pf::E16Part<BF> e;
	e.part = part;
	e.ld = N + Nd;
	e.kstride = (size_t)((M + 15) / 16 * 16) * (N + Nd);
	e.M = M;
	e.mul = BMAP::COLS_PER_TILE_DIV;
	if (s.bn == 256)
		return launch_g8p<pf::E16Part<BF>, BMAP, 2, 2>(f, A, lda, M, K, kb, bm, N + Nd, e, st, 0, Nd ? N : -1, Kd, s.nkc);
	if constexpr (BMAP::COLS_PER_TILE_DIV == 1) {
		if (s.bn == 192)
			return launch_g8p<pf::E16Part<BF>, BMAP, 2, 1>(f, A, lda, M, K, kb, bm, N + Nd, e, st, 0, Nd ? N : -1, Kd, s.nkc);
		return launch_g8p<pf::E16Part<BF>, BMAP, 1, 1>(f, A, lda, M, K, kb, bm, N + Nd, e, st, 0, Nd ? N : -1, Kd, s.nkc);
	}
	set_err("prefill GEMM: a gated pair's K slices have width 256");
	return YALM_ERR_UNSUPPORTED;
}

// c_split / K2: columns [c_split, N) run K2 (gemm8p_kernel); c_split = N: one depth
template <class EPI, class BMAP, int FJ0, int FJ1>
int launch_g8p(const PfForms &f, const uint16_t *A, int lda, int M, int K, int kb, const BMAP &bm, int N,
               const EPI &epi, hipStream_t st, int c0, int c_split, int K2, int nkc) {
	auto kern = pf::gemm8p_kernel<EPI, BMAP, FJ0, FJ1>;
	constexpr size_t lds = pf::gemm8p_lds<FJ0, FJ1, sizeof(pf::bmap_elt<BMAP>)>();
	constexpr int BN = 64 * (FJ0 + FJ1);
	static bool attr = false;
	if (!attr) {
		HIPCHK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
		attr = true;
	}
	const int tiles_m = (M + pf::G_BM - 1) / pf::G_BM;
	// (two depths: one workgroup per tile, so the hardware balances them longest first)
	const bool two = c_split >= 0 && c_split < N;
	const int ks1 = pf::epi_partial<EPI>::value ? slices(K, nkc) : 1, ks2 = pf::epi_partial<EPI>::value && two ? slices(K2, nkc) : 1;
	const int nwg = tiles_m * ((two ? c_split : N) / BN * ks1 + (two ? N - c_split : 0) / BN * ks2);
	// more tiles than CUs: one persistent workgroup per CU walks them
	const int ncu = (int)device_cu_count();
	const int grid = f.persist && nwg > ncu && !two && !pf::epi_partial<EPI>::value ? ncu : nwg;
	hipLaunchKernelGGL(kern, dim3(grid), dim3(pf::G_THREADS), lds, st, A, lda, M, K, kb, bm, N, epi, c0,
	                   two ? c_split : N, two ? K2 : K, nkc, pf::GrpNone{});
	HIPCHK(hipGetLastError());
	return YALM_OK;
}

// C[:, c0 .. c0 + N) = A · B^T over K columns of A (row stride lda) against B rows kb
// wide (K > kb: B wrap, prefill_gemm.h), tile 256 x BN
template <class EPI, class BMAP, int BN, int WM>
int launch_g16_t(const PfForms &f, const uint16_t *A, int lda, int M, int K, int kb, const BMAP &bm, int N,
                 const EPI &epi, hipStream_t st, int c0 = 0) {
	if (f.p8) { // the 8-phase schedule at the same tile width (320: spills, stays 2-phase)
		if constexpr (BN == 256 && WM == 2)
			return launch_g8p<EPI, BMAP, 2, 2>(f, A, lda, M, K, kb, bm, N, epi, st, c0);
		if constexpr (BN == 192 && WM == 2)
			return launch_g8p<EPI, BMAP, 2, 1>(f, A, lda, M, K, kb, bm, N, epi, st, c0);
		if constexpr (BN == 128 && BMAP::COLS_PER_TILE_DIV == 1) // GLU rows pair per 64-col wave
			return launch_g8p<EPI, BMAP, 1, 1>(f, A, lda, M, K, kb, bm, N, epi, st, c0);
	}
	if constexpr (sizeof(pf::bmap_elt<BMAP>) == 1) {
		set_err("prefill GEMM: E5M2 weights run on the 8-phase kernel (widths 128, 192, 256)");
		return YALM_ERR_UNSUPPORTED;
	} else {
		auto kern = pf::gemm16_kernel<EPI, BMAP, BN, WM>;
		constexpr size_t lds = pf::gemm16_lds<BN>();
		static bool attr = false;
		if (!attr) {
			HIPCHK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
			attr = true;
		}
		const int nwg = ((M + pf::G_BM - 1) / pf::G_BM) * (N / BN);
		hipLaunchKernelGGL(kern, dim3(nwg), dim3(pf::G_THREADS), lds, st, A, lda, M, K, kb, bm, N, epi, c0);
		HIPCHK(hipGetLastError());
		return YALM_OK;
	}
}

// C = A · W^T through the large-tile kernel at width bn (pick_bn; 0: no width fits)
template <class EPI, class BMAP>
int launch_rows(const PfForms &f, int bn, const uint16_t *A, int lda, int M, int K, int kb, const BMAP &bm, int N,
                const EPI &epi, hipStream_t st, int c0 = 0) {
	switch (bn) {
	case 128:
		return launch_g16_t<EPI, BMAP, 128, 4>(f, A, lda, M, K, kb, bm, N, epi, st, c0);
	case 192:
		return launch_g16_t<EPI, BMAP, 192, 2>(f, A, lda, M, K, kb, bm, N, epi, st, c0);
	case 256:
		return launch_g16_t<EPI, BMAP, 256, 2>(f, A, lda, M, K, kb, bm, N, epi, st, c0);
	case 320:
		return launch_g16_t<EPI, BMAP, 320, 2>(f, A, lda, M, K, kb, bm, N, epi, st, c0);
	}
	set_err("prefill GEMM: no 256-row tile width (128 / 192 / 256 / 320) divides N, or the forced one does not");
	return YALM_ERR_UNSUPPORTED;
}

// Weight rows from up to 3 matrices laid end to end: f16, or E5M2 bytes read as they are (e5m2)
struct WSrc {
	const void *p[3];
	int end[3];
	bool e5m2;
};
template <class F>
int with_rows(const WSrc &b, F launch) {
	if (b.e5m2) {
		pf::BRowsPlain8 r;
		for (int i = 0; i < 3; ++i)
			r.p[i] = (const uint8_t *)b.p[i], r.end[i] = b.end[i];
		return launch(r);
	}
	pf::BRowsPlain r;
	for (int i = 0; i < 3; ++i)
		r.src.p[i] = (const uint16_t *)b.p[i], r.src.end[i] = b.end[i];
	return launch(r);
}
// ... and a gated pair's two matrices
template <class F>
int with_glu(const void *w1, const void *w3, bool e5m2, F launch) {
	if (e5m2)
		return launch(pf::BRowsGlu<64, uint8_t>{(const uint8_t *)w1, (const uint8_t *)w3});
	return launch(pf::BRowsGlu<64>{(const uint16_t *)w1, (const uint16_t *)w3});
}
template <class EPI>
int launch_plain(const PfForms &f, int bn, const uint16_t *A, int lda, int M, int K, int kb, const WSrc &b,
                 int N, const EPI &epi, hipStream_t st, int c0 = 0) {
	return with_rows(b, [&](const auto &bm) { return launch_rows(f, bn, A, lda, M, K, kb, bm, N, epi, st, c0); });
}

// ---- short prompts (T <= SK_MAX_T): streamed GEMMs (prefill_skinny.h)
constexpr int SK_MAX_T = 64;
// rows of a streamed GEMM: 16, 32 (4 waves of 16 weight rows, two workgroups per CU) or 64 (8 waves, one)
int sk_rows(int T) { return T <= 16 ? 16 : T <= 32 ? 32 : 64; }
int sk_cols(int T) { return T <= 32 ? 64 : 128; }

// K slices of a streamed GEMM of N columns over nst stages of 128: ks slices of nsc stages. Rounds of the
// workgroups that fit the chip at once, a stage costing its share of HBM (2 x 16 KB or 32 KB of a CU's 26
// GB/ms, 1.27 us with every CU busy) or, with few workgroups, the latency behind its ring (0.7 us), 2 us to
// fill the ring, and for several slices a second launch that reads the partials (cap floats). The same for
// f16 and E5M2 weights, so an fp8 model sums in its f16 twin's order.
struct StreamPlan {
	int ks = 0, nsc = 0;
};
StreamPlan plan_stream(int T, int N, int nst, size_t cap) {
	const int blocks = (N + sk_cols(T) - 1) / sk_cols(T), rows = sk_rows(T);
	const float slots = (float)device_cu_count() * (T <= 32 ? 2 : 1);
	StreamPlan best;
	float least = 0.0f;
	for (int ks = 1; ks <= 16 && ks <= nst; ++ks) {
		const int nsc = (nst + ks - 1) / ks, k = (nst + nsc - 1) / nsc;
		const size_t floats = (size_t)k * rows * blocks * sk_cols(T);
		if (k != ks || (ks > 1 && (nsc < 2 || floats > cap)))
			continue;
		const float items = (float)blocks * ks;
		float t = std::ceil(items / slots) * (nsc * std::max(0.7f, 1.27f * std::min(1.0f, items / slots)) + 2.0f);
		if (ks > 1)
			t += 4.0f + (float)floats * 8.0f / 5e6f;
		if (!best.ks || t < least) {
			least = t;
			best = {ks, nsc};
		}
	}
	return best;
}

// GLU: over BRowsGlu rows (N = 2 x hidden, the epilogue's columns are hidden units). plan.ks == 1: the epilogue
// runs in the launch, else partials for launch_skinny_reduce / launch_reduce_norm. DUAL: columns >= c_split
// over [hi | lo].
template <int MT, int NW, class BMAP, bool DUAL, bool GLU, class EPI, bool BF>
int launch_stream_t(const PfForms &f, const StreamPlan &p, const uint16_t *A, int lda, int T, int K, int kb, const BMAP &bm,
                    int N, int c_split, float *part, const EPI &epi, hipStream_t st) {
	using C = pf::StreamCfg<MT, NW, BMAP, DUAL>;
	auto kern = pf::stream_gemm_kernel<MT, NW, BMAP, DUAL, GLU, EPI, BF>;
	static bool attr = false;
	if (!attr) {
		HIPCHK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS));
		attr = true;
	}
	const int nblk = (N + 16 * NW - 1) / (16 * NW);
	hipLaunchKernelGGL(kern, dim3(nblk * p.ks), dim3(64 * NW), C::LDS, st, A, lda, T, K / C::KSTG, kb, bm, nblk, p.nsc,
	                   c_split, nblk * 16 * NW, part, epi, (int)!f.skl);
	HIPCHK(hipGetLastError());
	return YALM_OK;
}
template <bool DUAL, bool GLU, bool BF, class BMAP, class EPI>
int launch_stream(const PfForms &f, const StreamPlan &p, const uint16_t *A, int lda, int T, int K, int kb, const BMAP &bm,
                  int N, int c_split, float *part, const EPI &epi, hipStream_t st) {
	if (T <= 16)
		return launch_stream_t<1, 4, BMAP, DUAL, GLU, EPI, BF>(f, p, A, lda, T, K, kb, bm, N, c_split, part, epi, st);
	if (T <= 32)
		return launch_stream_t<2, 4, BMAP, DUAL, GLU, EPI, BF>(f, p, A, lda, T, K, kb, bm, N, c_split, part, epi, st);
	return launch_stream_t<4, 8, BMAP, DUAL, GLU, EPI, BF>(f, p, A, lda, T, K, kb, bm, N, c_split, part, epi, st);
}

// columns < c_split sum KS partials, the others KS2
template <bool GLU, class EPI>
int launch_skinny_reduce(const float *part, int KS, int KS2, int c_split, int T, int Np, const EPI &epi,
                         hipStream_t st, int TP = 0) { // TP: rows of a slot (default: T in whole 16s)
	TP = TP ? TP : 16 * ((T + 15) / 16);
	const int waves = ((T + 15) / 16) * (Np / 64);
	pf::skinny_reduce_kernel<4, GLU, EPI><<<(waves + 3) / 4, 256, 0, st>>>(part, KS, KS2, c_split, TP, T, Np, epi);
	HIPCHK(hipGetLastError());
	return YALM_OK;
}

WSrc one(const void *w, int rows, bool e5m2 = false) { return WSrc{{w, w, w}, {rows, rows, rows}, e5m2}; }

// fp8 models in the forms that cannot read the bytes (yalm_set_prefill_forms' other tilings, a classifier of
// width-320 tiles): the tensors (E5M2 bytes, n elements each) dequantised to f16 into b.wdq, end
// to end; returns their f16 copies in `out` (prefill.h e5m2_to_f16_kernel)
int dequant(yalm_decoder_s *d, std::initializer_list<std::pair<const void *, size_t>> t, const uint16_t **out,
			hipStream_t st) {
	if (!d->pf.wdq) { // one layer's weights, or the classifier's
		const yalm_config &c = d->c;
		const size_t q_dim = (size_t)c.n_heads * c.head_dim;
		const size_t layer = (q_dim + 2 * (size_t)c.n_kv_heads * c.head_dim) * c.dim + (size_t)c.dim * q_dim +
							 3 * (size_t)c.dim * c.hidden_dim;
		TRY(pf_alloc(d, (void **)&d->pf.wdq, 2 * std::max(layer, (size_t)c.vocab_size * c.dim)));
	}
	pf::DqSegs s{};
	size_t off = 0, pieces = 0;
	for (auto &p : t) {
		s.src[s.n] = (const uint8_t *)p.first;
		s.dst[s.n] = d->pf.wdq + off;
		out[s.n] = s.dst[s.n];
		pieces += p.second / 16;
		s.end[s.n] = pieces;
		off += p.second;
		++s.n;
	}
	const int grid = (int)std::min<size_t>((pieces + 255) / 256, (size_t)device_cu_count() * 8);
	pf::e5m2_to_f16_kernel<<<grid, 256, 0, st>>>(s);
	HIPCHK(hipGetLastError());
	return YALM_OK;
}

// Xn = f16(rmsnorm(X) * w) rows (SPLIT: [hi | lo]): one wave per row with the row in
// registers (prefill.h rmsnorm_rows_wave_kernel) when dim <= 8192, else (or forms "wnorm:0")
// the workgroup-per-row kernel
template <bool SPLIT>
int launch_rmsnorm_t(const PfForms &f, const float *X, const float *w, int dim, int T, float eps, uint16_t *Xn,
                     unsigned *range, hipStream_t st) {
	const int nv = (dim / 4 + 63) / 64; // float4 per lane
	const int g = (T + 3) / 4;
	if (f.wnorm && nv <= 32) {
		if (nv <= 4)
			pf::rmsnorm_rows_wave_kernel<SPLIT, 4><<<g, 256, 0, st>>>(X, w, dim, T, eps, Xn, range);
		else if (nv <= 8)
			pf::rmsnorm_rows_wave_kernel<SPLIT, 8><<<g, 256, 0, st>>>(X, w, dim, T, eps, Xn, range);
		else if (nv <= 12)
			pf::rmsnorm_rows_wave_kernel<SPLIT, 12><<<g, 256, 0, st>>>(X, w, dim, T, eps, Xn, range);
		else if (nv <= 16)
			pf::rmsnorm_rows_wave_kernel<SPLIT, 16><<<g, 256, 0, st>>>(X, w, dim, T, eps, Xn, range);
		else if (nv <= 24)
			pf::rmsnorm_rows_wave_kernel<SPLIT, 24><<<g, 256, 0, st>>>(X, w, dim, T, eps, Xn, range);
		else
			pf::rmsnorm_rows_wave_kernel<SPLIT, 32><<<g, 256, 0, st>>>(X, w, dim, T, eps, Xn, range);
	} else {
		pf::rmsnorm_rows_kernel<SPLIT><<<T, 256, 0, st>>>(X, w, dim, eps, Xn, range);
	}
	HIPCHK(hipGetLastError());
	return YALM_OK;
}
int launch_rmsnorm(bool split, const PfForms &f, const float *X, const float *w, int dim, int T, float eps, uint16_t *Xn,
                   unsigned *range, hipStream_t st) {
	return split ? launch_rmsnorm_t<true>(f, X, w, dim, T, eps, Xn, range, st)
	             : launch_rmsnorm_t<false>(f, X, w, dim, T, eps, Xn, range, st);
}

// X += scale * (sum of the partials), Xn = the next norm's operand (prefill_skinny.h); w null: no norm
template <bool SPLIT>
int launch_reduce_norm_t(const float *part, int KS, int T, float *X, int dim, float scale, const float *w, float eps,
                         uint16_t *Xn, unsigned *range, hipStream_t st, int TP) {
	const size_t kstride = (size_t)TP * dim;
	const int nt = std::min(1024, (dim / 4 + 63) / 64 * 64), nv = (dim / 4 + nt - 1) / nt;
	if (nv == 1)
		pf::reduce_norm_rows_kernel<SPLIT, 1><<<T, nt, 0, st>>>(part, KS, kstride, X, dim, scale, w, eps, Xn, range);
	else if (nv == 2)
		pf::reduce_norm_rows_kernel<SPLIT, 2><<<T, nt, 0, st>>>(part, KS, kstride, X, dim, scale, w, eps, Xn, range);
	else
		pf::reduce_norm_rows_kernel<SPLIT, 4><<<T, nt, 0, st>>>(part, KS, kstride, X, dim, scale, w, eps, Xn, range);
	HIPCHK(hipGetLastError());
	return YALM_OK;
}
int launch_reduce_norm(bool split, const float *part, int KS, int T, float *X, int dim, float scale, const float *w,
                       float eps, uint16_t *Xn, unsigned *range, hipStream_t st, int TP) {
	return split ? launch_reduce_norm_t<true>(part, KS, T, X, dim, scale, w, eps, Xn, range, st, TP)
	             : launch_reduce_norm_t<false>(part, KS, T, X, dim, scale, w, eps, Xn, range, st, TP);
}
constexpr int REDUCE_NORM_MAX_DIM = 4 * 1024 * 4; // the row in registers: 4 float4 of 1024 threads

template <int D, bool SPLIT>
int launch_attn_prefill_t(const uint16_t *Q, const uint16_t *kc, const uint16_t *vc, int T, int pos0, int n_heads,
						  int n_kv, uint16_t *O, hipStream_t st) {
	const dim3 grid(n_heads, (T + pf::AQ - 1) / pf::AQ); // heads fastest: longest-first dispatch
	auto kern = pf::attn_prefill_kernel<D, pf::AKT, SPLIT>;
	static bool attr_set = false;
	if (!attr_set) {
		HIPCHK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
								   (int)pf::attn_prefill_lds<D>()));
		attr_set = true;
	}
	hipLaunchKernelGGL(kern, grid, dim3(pf::THREADS), pf::attn_prefill_lds<D>(), st, Q, kc, vc, T, pos0, n_heads, n_kv,
					   O);
	HIPCHK(hipGetLastError());
	return YALM_OK;
}

// split: Q and O rows [hi | lo] (the split-operand form)
int launch_attn_prefill(const uint16_t *Q, const uint16_t *kc, const uint16_t *vc, int T, int pos0, int n_heads,
						int n_kv, int head_dim, uint16_t *O, hipStream_t st, bool split = false) {
	if (head_dim == 128)
		return split ? launch_attn_prefill_t<128, true>(Q, kc, vc, T, pos0, n_heads, n_kv, O, st)
					 : launch_attn_prefill_t<128, false>(Q, kc, vc, T, pos0, n_heads, n_kv, O, st);
	if (head_dim == 64)
		return split ? launch_attn_prefill_t<64, true>(Q, kc, vc, T, pos0, n_heads, n_kv, O, st)
					 : launch_attn_prefill_t<64, false>(Q, kc, vc, T, pos0, n_heads, n_kv, O, st);
	set_err("prefill attention: head_dim must be 64 or 128");
	return YALM_ERR_UNSUPPORTED;
}

int check_prefill_shape(const yalm_config &c) {
	const int q_dim = c.n_heads * c.head_dim, kv_dim = c.n_kv_heads * c.head_dim;
	if (c.weight_dtype != YALM_F16 && c.weight_dtype != YALM_F8E5M2) {
		set_err("yalm_prefill: f16 or fp8 (E5M2) weights only (MFMA f16 operands)");
		return YALM_ERR_UNSUPPORTED;
	}
	if (c.dim % pf::BN || c.hidden_dim % pf::BN || q_dim % pf::BN || kv_dim % pf::BN || c.vocab_size % pf::BN ||
	    (c.head_dim != 64 && c.head_dim != 128)) {
		set_err("yalm_prefill: dims must be multiples of 128 and head_dim 64 or 128");
		return YALM_ERR_UNSUPPORTED;
	}
	return YALM_OK;
}

int ensure_bufs(yalm_decoder_s *d) {
	PrefillBufs &b = d->pf;
	if (b.cap)
		return YALM_OK;
	const yalm_config &c = d->c;
	const size_t cap = (size_t)c.max_seq_len, q_dim = (size_t)c.n_heads * c.head_dim;
	const size_t ntiles = (size_t)c.vocab_size / pf::BN;
	TRY(pf_alloc(d, (void **)&b.X, cap * c.dim * 4));
	TRY(pf_alloc(d, (void **)&b.Xn, cap * c.dim * 2 * 2));
	// Q, O, H: [hi | lo] rows in the split-operand form, 2x wide
	TRY(pf_alloc(d, (void **)&b.Q, cap * q_dim * 2 * 2));
	TRY(pf_alloc(d, (void **)&b.O, cap * q_dim * 2 * 2));
	TRY(pf_alloc(d, (void **)&b.H, cap * c.hidden_dim * 2 * 2));
	TRY(pf_alloc(d, (void **)&b.tok, cap * 4));
	TRY(pf_alloc(d, (void **)&b.tgt, cap * 4));
	TRY(pf_alloc(d, (void **)&b.pmax, cap * ntiles * 4));
	TRY(pf_alloc(d, (void **)&b.psum, cap * ntiles * 4));
	TRY(pf_alloc(d, (void **)&b.tgt_logit, cap * 4));
	TRY(pf_alloc(d, (void **)&b.lp, cap * 4));
	TRY(pf_alloc(d, (void **)&b.rope, cap * c.head_dim * 4));
	TRY(pf_alloc(d, (void **)&b.range, (size_t)(c.n_layers + 1) * RG_N * 4));
	{ // f32 partials of K slices, at most 128 MB: plan_split and plan_stream keep to it
		const size_t widest = std::max({q_dim + 2 * (size_t)c.n_kv_heads * c.head_dim, (size_t)c.dim, (size_t)2 * c.hidden_dim});
		b.skp_floats = std::min((size_t)32 << 20, 16 * std::max((cap + 15) / 16 * 16, (size_t)SK_MAX_T) * (widest + 64));
		TRY(pf_alloc(d, (void **)&b.skp, b.skp_floats * 4));
	}
	b.cap = (int)cap;
	return YALM_OK;
}

template <int ACT, bool SPLIT>
int enqueue_glu_t(yalm_decoder_s *d, const yalm_block_weights &w, int T, float hscale, unsigned *range, bool e5m2) {
	const yalm_config &c = d->c;
	const PfForms &f = d->pf_forms;
	const int bn = pick_bn(f, PG_GLU, T, 2 * c.hidden_dim, true, false, e5m2);
	const int sp = SPLIT ? 2 : 1; // split-operand form: A = [hi | lo] (K = 2 dim), H rows [hi | lo]
	pf::E16Glu<ACT, SPLIT> e;
	e.h = d->pf.H;
	e.ldh = c.hidden_dim * sp;
	e.M = T;
	e.hscale = hscale;
	e.range = range;
	e.lo_off = SPLIT ? c.hidden_dim : 0;
	const SplitPlan s = plan_split(f, PG_GLU, T, 2 * c.hidden_dim, sp * c.dim, 0, 0, true, d->pf.skp_floats);
	return with_glu(w.w1, w.w3, e5m2, [&](const auto &bm) -> int {
		using BM = std::decay_t<decltype(bm)>;
		if (s.ks > 1) {
			TRY(launch_split(f, s, d->pf.Xn, sp * c.dim, T, sp * c.dim, c.dim, bm, 2 * c.hidden_dim, 0, 0, d->pf.skp, d->stream));
			return launch_skinny_reduce<true>(d->pf.skp, s.ks, s.ks, 2 * c.hidden_dim, T, 2 * c.hidden_dim, e, d->stream);
		}
		if (bn == 256)
			return launch_g16_t<pf::E16Glu<ACT, SPLIT>, BM, 256, 2>(f, d->pf.Xn, sp * c.dim, T, sp * c.dim, c.dim, bm,
			                                                        2 * c.hidden_dim, e, d->stream);
		if (bn == 128)
			return launch_g16_t<pf::E16Glu<ACT, SPLIT>, BM, 128, 4>(f, d->pf.Xn, sp * c.dim, T, sp * c.dim, c.dim, bm,
			                                                        2 * c.hidden_dim, e, d->stream);
		set_err("prefill GLU GEMM: 2 x hidden_dim must divide by 128 (or by a forced width of 128 / 256)");
		return YALM_ERR_UNSUPPORTED;
	});
}

template <int ACT>
int enqueue_glu(yalm_decoder_s *d, const yalm_block_weights &w, int T, float hscale, unsigned *range, bool e5m2) {
	return d->pf_forms.split ? enqueue_glu_t<ACT, true>(d, w, T, hscale, range, e5m2)
	                         : enqueue_glu_t<ACT, false>(d, w, T, hscale, range, e5m2);
}

// The whole prefill on d->stream: T rows at positions pos0 .. pos0 + T - 1. hexp[l] (null:
// all 0): layer l's GLU output is stored as f16(h * 2^-hexp[l]) and W2 adds 2^hexp[l] x its
// product (exact power-of-two scales; yalm_prefill chooses them from the range guard).
int enqueue_prefill(yalm_decoder_s *d, int T, int pos0, bool want_lp, const int *hexp = nullptr) {
	const yalm_config &c = d->c;
	const PfForms &f = d->pf_forms;
	PrefillBufs &b = d->pf;
	hipStream_t st = d->stream;
	const int q_dim = c.n_heads * c.head_dim, kv_dim = c.n_kv_heads * c.head_dim;
	const bool fp8 = c.weight_dtype == YALM_F8E5M2;
	if (fp8)
		pf::embed_rows_kernel<WF8><<<T, 256, 0, st>>>(b.tok, d->emb, c.dim, b.X);
	else
		pf::embed_rows_kernel<WF16><<<T, 256, 0, st>>>(b.tok, d->emb, c.dim, b.X);
	HIPCHK(hipGetLastError());
	const int half = c.head_dim / 2;
	pf::rope_table_kernel<<<(T * half + 255) / 256, 256, 0, st>>>(d->inv_freq, half, T, pos0, b.rope);
	HIPCHK(hipGetLastError());
	// fp8: every GEMM reads the E5M2 bytes (gemm8p_kernel, stream_gemm_kernel) with the slices and K order of
	// the f16 twin, so the results are its bit for bit; forms that name other kernels run on f16 copies
	const bool raw8 = fp8 && f.p8 && f.skl && f.g16[PG_QKV] < 0 && f.g16[PG_WO] < 0 && f.g16[PG_GLU] < 0 && f.g16[PG_W2] < 0;
	// GEMM widths are the same for every layer
	const int bn_q = pick_bn(f, PG_QKV, T, q_dim, false, false, raw8);
	const int bn_kv = pick_bn(f, PG_QKV, T, 2 * kv_dim, false, false, raw8);
	// q and k | v in one two-depth launch at width 256 (gemm8p_kernel): the two launches'
	// tiles balanced over the chip instead of one round each (Llama-3B at T 4096: q 82 us
	// at width 192 + k | v 115 us at 128)
	const bool qkv1 = f.qkv1 && f.p8 && f.g16[PG_QKV] < 0 && q_dim % 256 == 0 && (2 * kv_dim) % 256 == 0;
	const int bn_wo = pick_bn(f, PG_WO, T, c.dim, false, false, raw8);
	const int bn_w2 = pick_bn(f, PG_W2, T, c.dim, false, false, raw8);
	// short prompts: streamed GEMMs (the 256-row tiles would leave most CUs idle)
	const bool small = T <= SK_MAX_T && !f.no_skinny && !f.split;
	const int TP = small ? sk_rows(T) : (T + 15) / 16 * 16; // rows of a partial slot
	const int nstg = pf::StreamCfg<1, 4, pf::BRowsPlain, false>::KSTG;
	const StreamPlan p_qkv = plan_stream(T, q_dim + 2 * kv_dim, c.dim / nstg, b.skp_floats);
	const StreamPlan p_wo = plan_stream(T, c.dim, q_dim / nstg, b.skp_floats);
	const StreamPlan p_glu = plan_stream(T, 2 * c.hidden_dim, c.dim / nstg, b.skp_floats);
	const StreamPlan p_w2 = plan_stream(T, c.dim, c.hidden_dim / nstg, b.skp_floats);
	// the split-operand precision form (yalm_set_prefill_precision): every activation operand
	// [hi | lo] -- the normalised x of all three norms, Q, P (attention.h SPLIT), O and H --
	// each GEMM over K = 2 x its depth with the B rows wrapping (prefill_gemm.h), so no operand
	// carries an f16 rounding the reference's f32 lacks; sp = operand width factor
	const bool split = f.split;
	const int sp = split ? 2 : 1;
	const int bn_qkv_all = pick_bn(f, PG_QKV, T, q_dim + 2 * kv_dim, false, false, raw8);
	// too few tiles for the chip: K slices. Wo's and W2's partials, and a short prompt's, are
	// summed by the launch that also adds the residual and makes the next product's operand
	const size_t pcap = b.skp_floats;
	const SplitPlan s_qkv = split ? plan_split(f, PG_QKV, T, q_dim + 2 * kv_dim, 2 * c.dim, 0, 0, false, pcap)
	                              : plan_split(f, PG_QKV, T, q_dim, c.dim, 2 * kv_dim, 2 * c.dim, false, pcap);
	const SplitPlan s_wo = plan_split(f, PG_WO, T, c.dim, sp * q_dim, 0, 0, false, pcap);
	const SplitPlan s_w2 = plan_split(f, PG_W2, T, c.dim, sp * c.hidden_dim, 0, 0, false, pcap);
	const bool fused_norm = f.wnorm && c.dim <= REDUCE_NORM_MAX_DIM;
	auto reduce_norm = [&](int KS, float scale, const float *w, bool xsplit, unsigned *range) -> int {
		if (!fused_norm) { // (rows too wide for the fused kernel's registers)
			pf::E16Residual e;
			e.x = b.X, e.ldx = c.dim, e.M = T, e.scale = scale;
			TRY(launch_skinny_reduce<false>(b.skp, KS, KS, c.dim, T, c.dim, e, st, TP));
			return w ? launch_rmsnorm(xsplit, f, b.X, w, c.dim, T, c.norm_eps, b.Xn, range, st) : YALM_OK;
		}
		return launch_reduce_norm(xsplit, b.skp, KS, T, b.X, c.dim, scale, w, c.norm_eps, b.Xn, range, st, TP);
	};
	// a streamed product: one slice runs the epilogue itself, several leave partials to be reduced
	auto stream = [&](auto DUALc, auto GLUc, const StreamPlan &p, const uint16_t *A, int lda, int K, const auto &bm, int N,
	                  int c_split, const auto &e) -> int {
		constexpr bool DUAL = decltype(DUALc)::value, GLU = decltype(GLUc)::value;
		if (p.ks == 1)
			return launch_stream<DUAL, GLU, false>(f, p, A, lda, T, K, K, bm, N, c_split, nullptr, e, st);
		TRY((launch_stream<DUAL, GLU, false>(f, p, A, lda, T, K, K, bm, N, c_split, b.skp, pf::NoEpi{}, st)));
		return launch_skinny_reduce<GLU>(b.skp, p.ks, p.ks, N, T, N, e, st, TP);
	};
	bool normed = false; // Xn holds this layer's attention input already
	for (int l = 0; l < c.n_layers; ++l) {
		yalm_block_weights w = d->b[l];
		if (fp8 && !raw8) { // this layer's weights as f16 (exact), in the scratch the previous layer's GEMMs are done with
			const uint16_t *p[7];
			const size_t qd = (size_t)q_dim * c.dim, kd = (size_t)kv_dim * c.dim, hd = (size_t)c.hidden_dim * c.dim;
			TRY(dequant(d, {{w.wq, qd}, {w.wk, kd}, {w.wv, kd}, {w.wo, qd}, {w.w1, hd}, {w.w2, hd}, {w.w3, hd}}, p, st));
			w.wq = p[0], w.wk = p[1], w.wv = p[2], w.wo = p[3], w.w1 = p[4], w.w2 = p[5], w.w3 = p[6];
		}
		// normalised x as [hi | lo] (2 dim per row): hi is the q columns' A operand, hi + lo
		// the k | v columns' (their cache rows then carry one f16 rounding, infer.cpp:299)
		unsigned *rg = b.range + (size_t)l * RG_N;
		const int he = hexp ? hexp[l] : 0;
		if (!normed)
			TRY(launch_rmsnorm(true, f, b.X, w.rms_att, c.dim, T, c.norm_eps, b.Xn, rg + RG_XATT, st));
		{
			const WSrc qkv{{w.wq, w.wk, w.wv}, {q_dim, q_dim + kv_dim, q_dim + 2 * kv_dim}, raw8};
			pf::E16QKV e;
			e.q = b.Q;
			e.kc = w.key_cache;
			e.vc = w.value_cache;
			e.rope = b.rope;
			e.M = T;
			e.q_dim = q_dim;
			e.kv_dim = kv_dim;
			e.head_dim = c.head_dim;
			e.pos0 = pos0;
			e.clip = c.qkv_clip;
			e.range = rg + RG_Q;
			// QKV + clip + RoPE as two GEMMs: q (K = dim over hi) and k | v from column
			// q_dim (K = 2 dim over hi | lo, the B rows wrapping at dim)
			if (small) {
				// one launch: q over hi, k | v over [hi | lo]
				TRY(with_rows(qkv, [&](const auto &bm) {
					return stream(std::true_type{}, std::false_type{}, p_qkv, b.Xn, 2 * c.dim, c.dim, bm, q_dim + 2 * kv_dim, q_dim, e);
				}));
			} else {
				const int np = q_dim + 2 * kv_dim;
				if (split) { // q | k | v all over [hi | lo], Q stored [hi | lo]
					pf::E16QKVt<true> es;
					es.q = e.q, es.kc = e.kc, es.vc = e.vc, es.rope = e.rope, es.M = e.M, es.q_dim = e.q_dim;
					es.kv_dim = e.kv_dim, es.head_dim = e.head_dim, es.pos0 = e.pos0, es.clip = e.clip;
					es.range = e.range, es.q_lo = q_dim;
					if (s_qkv.ks > 1) {
						TRY(with_rows(qkv, [&](const auto &bm) {
							return launch_split(f, s_qkv, b.Xn, 2 * c.dim, T, 2 * c.dim, c.dim, bm, np, 0, 0, b.skp, st);
						}));
						TRY(launch_skinny_reduce<false>(b.skp, s_qkv.ks, s_qkv.ks, np, T, np, es, st));
					} else {
						TRY(launch_plain(f, bn_qkv_all, b.Xn, 2 * c.dim, T, 2 * c.dim, c.dim, qkv, np, es, st));
					}
				} else if (s_qkv.ks > 1) {
					TRY(with_rows(qkv, [&](const auto &bm) {
						return launch_split(f, s_qkv, b.Xn, 2 * c.dim, T, c.dim, c.dim, bm, q_dim, 2 * kv_dim, 2 * c.dim, b.skp, st);
					}));
					TRY(launch_skinny_reduce<false>(b.skp, s_qkv.ks, s_qkv.ks2, q_dim, T, np, e, st));
				} else if (qkv1) { // one launch: the k | v tiles (K = 2 dim) first, then the q tiles (K = dim)
					TRY(with_rows(qkv, [&](const auto &bm) {
						return launch_g8p<pf::E16QKV, std::decay_t<decltype(bm)>, 2, 2>(
						    f, b.Xn, 2 * c.dim, T, c.dim, c.dim, bm, q_dim + 2 * kv_dim, e, st, 0, q_dim, 2 * c.dim);
					}));
				} else {
					TRY(launch_plain(f, bn_q, b.Xn, 2 * c.dim, T, c.dim, c.dim, qkv, q_dim, e, st));
					TRY(launch_plain(f, bn_kv, b.Xn, 2 * c.dim, T, 2 * c.dim, c.dim, qkv, 2 * kv_dim, e, st, q_dim));
				}
			}
		}
		TRY(launch_attn_prefill(b.Q, w.key_cache, w.value_cache, T, pos0, c.n_heads, c.n_kv_heads, c.head_dim, b.O,
								st, split));
		if (small || s_wo.ks > 1) {
			TRY(with_rows(one(w.wo, c.dim, raw8), [&](const auto &bm) {
				return small ? launch_stream<false, false, false>(f, p_wo, b.O, q_dim, T, q_dim, q_dim, bm, c.dim, c.dim, b.skp,
				                                                  pf::NoEpi{}, st)
				             : launch_split(f, s_wo, b.O, sp * q_dim, T, sp * q_dim, q_dim, bm, c.dim, 0, 0, b.skp, st);
			}));
			TRY(reduce_norm(small ? p_wo.ks : s_wo.ks, 1.0f, w.rms_ffn, split, rg + RG_XFFN));
		} else {
			pf::E16Residual e;
			e.x = b.X;
			e.ldx = c.dim;
			e.M = T;
			TRY(launch_plain(f, bn_wo, b.O, sp * q_dim, T, sp * q_dim, q_dim, one(w.wo, c.dim, raw8), c.dim, e, st));
			TRY(launch_rmsnorm(split, f, b.X, w.rms_ffn, c.dim, T, c.norm_eps, b.Xn, rg + RG_XFFN, st));
		}
		const float hscale = ldexpf(1.0f, -he);
		if (small) {
			auto glu = [&](auto e) -> int {
				e.h = b.H, e.ldh = c.hidden_dim, e.M = T, e.hscale = hscale, e.range = rg + RG_H;
				return with_glu(w.w1, w.w3, raw8, [&](const auto &bm) {
					return stream(std::false_type{}, std::true_type{}, p_glu, b.Xn, c.dim, c.dim, bm, 2 * c.hidden_dim, 2 * c.hidden_dim, e);
				});
			};
			TRY(c.act == YALM_SILU ? glu(pf::E16Glu<1>{}) : glu(pf::E16Glu<0>{}));
		} else {
			TRY(c.act == YALM_SILU ? enqueue_glu<1>(d, w, T, hscale, rg + RG_H, raw8)
								   : enqueue_glu<0>(d, w, T, hscale, rg + RG_H, raw8));
		}
		// the next norm: the next layer's (its operand [hi | lo] in either form), or the final one
		const bool last = l + 1 == c.n_layers;
		const float *w_next = last ? (want_lp ? d->rms_final : nullptr) : d->b[l + 1].rms_att;
		normed = small || s_w2.ks > 1;
		if (normed) {
			TRY(with_rows(one(w.w2, c.dim, raw8), [&](const auto &bm) {
				const int h = c.hidden_dim;
				return small ? launch_stream<false, false, false>(f, p_w2, b.H, h, T, h, h, bm, c.dim, c.dim, b.skp, pf::NoEpi{}, st)
				             : launch_split(f, s_w2, b.H, sp * h, T, sp * h, h, bm, c.dim, 0, 0, b.skp, st);
			}));
			TRY(reduce_norm(small ? p_w2.ks : s_w2.ks, ldexpf(1.0f, he), w_next, last ? split : true, rg + RG_N + RG_XATT));
		} else {
			pf::E16Residual e;
			e.x = b.X;
			e.ldx = c.dim;
			e.M = T;
			e.scale = ldexpf(1.0f, he);
			TRY(launch_plain(f, bn_w2, b.H, sp * c.hidden_dim, T, sp * c.hidden_dim, c.hidden_dim,
			                 one(w.w2, c.dim, raw8), c.dim, e, st));
		}
	}
	if (!want_lp)
		return YALM_OK;
	if (!normed)
		TRY(launch_rmsnorm(split, f, b.X, d->rms_final, c.dim, T, c.norm_eps, b.Xn,
		                   b.range + (size_t)c.n_layers * RG_N + RG_XATT, st));
	const int cls_bn = pick_bn(f, PG_CLS, T, c.vocab_size, false);
	const int ntiles = cls_bn ? c.vocab_size / cls_bn : 1;
	pf::E16Logits e;
	e.pmax = b.pmax;
	e.psum = b.psum;
	e.tgt_logit = b.tgt_logit;
	e.targets = b.tgt;
	e.M = T;
	e.ntiles = ntiles;
	e.red = nullptr;
	const void *wcls = d->wcls;
	const bool cls8 = raw8 && f.g16[PG_CLS] < 0 && cls_bn <= 256; // (the f16 twin's tile width decides the sums' order)
	if (fp8 && !cls8) {
		const uint16_t *p[1];
		TRY(dequant(d, {{d->wcls, (size_t)c.vocab_size * c.dim}}, p, st));
		wcls = p[0];
	}
	TRY(launch_plain(f, cls_bn, b.Xn, sp * c.dim, T, sp * c.dim, c.dim, one(wcls, c.vocab_size, cls8), c.vocab_size,
	                 e, st));
	pf::logprob_kernel<<<T, 256, 0, st>>>(b.pmax, b.psum, b.tgt_logit, b.tgt, T, ntiles, b.lp);
	HIPCHK(hipGetLastError());
	return YALM_OK;
}

struct HostDev { // scoped device copy for the test hooks
	void *p = nullptr;
	~HostDev() {
		if (p)
			(void)hipFree(p);
	}
};
int hd(HostDev &b, const void *host, size_t bytes) {
	HIPCHK(hipMalloc(&b.p, bytes ? bytes : 4));
	if (host)
		HIPCHK(hipMemcpy(b.p, host, bytes, hipMemcpyHostToDevice));
	else
		HIPCHK(hipMemset(b.p, 0, bytes));
	return YALM_OK;
}

} // namespace

extern "C" int yalm_prefill(yalm_decoder d, const int *tokens, int n, int pos0, float *logprobs) {
	ARGCHK(d && tokens && n > 0 && pos0 >= 0, "yalm_prefill: bad argument");
	const yalm_config &c = d->c;
	ARGCHK(pos0 + n <= c.max_seq_len, "yalm_prefill: pos0 + n must be <= max_seq_len (no sliding window in prefill)");
	TRY(check_prefill_shape(c));
	TRY(ensure_bufs(d));
	PrefillBufs &b = d->pf;
	std::vector<int> tgt(n);
	for (int i = 0; i < n; ++i) {
		ARGCHK(tokens[i] >= 0 && tokens[i] < c.vocab_size, "yalm_prefill: token id out of range");
		tgt[i] = i + 1 < n ? tokens[i + 1] : -1;
	}
	HIPCHK(hipMemcpyAsync(b.tok, tokens, sizeof(int) * n, hipMemcpyHostToDevice, d->stream));
	HIPCHK(hipMemcpyAsync(b.tgt, tgt.data(), sizeof(int) * n, hipMemcpyHostToDevice, d->stream));
	// The range guard (prefill.h range_note): a pass whose f16 operands all fit is the result.
	// Otherwise the FIRST slot out of range decides (everything after it saw inf / NaN): a GLU
	// output gets the exact power-of-two scale that brings its largest |h| under 2^14 and the
	// pass runs again (idempotent: the same cache rows and log-probs are rewritten); any
	// other operand out of range (the normalised x, Q, the final norm) is refused.
	const int L = c.n_layers;
	std::vector<int> hexp(L, 0);
	std::vector<unsigned> rg((size_t)(L + 1) * RG_N);
	b.last_passes = b.last_scaled = 0;
	for (int pass = 1;; ++pass) {
		HIPCHK(hipMemsetAsync(b.range, 0, rg.size() * 4, d->stream));
		TRY(enqueue_prefill(d, n, pos0, logprobs != nullptr, hexp.data()));
		HIPCHK(hipMemcpyAsync(rg.data(), b.range, rg.size() * 4, hipMemcpyDeviceToHost, d->stream));
		HIPCHK(hipStreamSynchronize(d->stream));
		b.last_passes = pass;
		int bad = -1;
		for (size_t i = 0; i < rg.size() && bad < 0; ++i)
			if (rg[i])
				bad = (int)i;
		if (bad < 0)
			break;
		const int l = bad / RG_N, kind = bad % RG_N;
		float mx;
		memcpy(&mx, &rg[bad], 4);
		static const char *what[RG_N] = {"the normalised x (attention input)", "Q", "the normalised x (FFN input)",
										 "the GLU output"};
		if (kind != RG_H || l >= L || !std::isfinite(mx) || pass > L + 1) {
			set_err(std::string("yalm_prefill: ") + (l >= L ? "the final norm's output" : what[kind]) + " of layer " +
					std::to_string(l) + " exceeds the f16 range of the MFMA operands (max |v| " +
					std::to_string(mx) + "); the decode path (yalm_forward) keeps it in f32");
			return YALM_ERR_UNSUPPORTED;
		}
		const int e = (int)std::ceil(std::log2(mx / 16384.0f));
		if (e <= hexp[l]) { // cannot happen for a finite max: a scale that did not help
			set_err("yalm_prefill: internal: the GLU output scale did not bring layer " + std::to_string(l) + " into range");
			return YALM_ERR_HIP;
		}
		hexp[l] = e;
	}
	for (int l = 0; l < L; ++l)
		b.last_scaled += hexp[l] > 0;
	if (logprobs)
		HIPCHK(hipMemcpy(logprobs, b.lp, sizeof(float) * n, hipMemcpyDeviceToHost));
	return YALM_OK;
}

extern "C" int yalm_prefill_info(yalm_decoder d, int *passes, int *scaled_layers) {
	ARGCHK(d, "null decoder");
	if (passes)
		*passes = d->pf.last_passes;
	if (scaled_layers)
		*scaled_layers = d->pf.last_scaled;
	return YALM_OK;
}

extern "C" int yalm_prefill_time(yalm_decoder d, int n, int iters, float *avg_ms) {
	ARGCHK(d && n > 0 && iters > 0 && avg_ms, "yalm_prefill_time: bad argument");
	const yalm_config &c = d->c;
	ARGCHK(n <= c.max_seq_len, "yalm_prefill_time: n > max_seq_len");
	TRY(check_prefill_shape(c));
	TRY(ensure_bufs(d));
	std::vector<int> tok(n);
	for (int i = 0; i < n; ++i)
		tok[i] = (int)((1103515245u * (unsigned)i + 12345u) % (unsigned)c.vocab_size);
	HIPCHK(hipMemcpy(d->pf.tok, tok.data(), sizeof(int) * n, hipMemcpyHostToDevice));
	for (int i = 0; i < n; ++i)
		tok[i] = i + 1 < n ? tok[i + 1] : -1;
	HIPCHK(hipMemcpy(d->pf.tgt, tok.data(), sizeof(int) * n, hipMemcpyHostToDevice));
	TRY(enqueue_prefill(d, n, 0, true)); // warm-up
	hipEvent_t e0, e1;
	HIPCHK(hipEventCreate(&e0));
	HIPCHK(hipEventCreate(&e1));
	HIPCHK(hipEventRecord(e0, d->stream));
	for (int i = 0; i < iters; ++i)
		TRY(enqueue_prefill(d, n, 0, true));
	HIPCHK(hipEventRecord(e1, d->stream));
	HIPCHK(hipEventSynchronize(e1));
	float ms = 0;
	HIPCHK(hipEventElapsedTime(&ms, e0, e1));
	(void)hipEventDestroy(e0);
	(void)hipEventDestroy(e1);
	*avg_ms = ms / iters;
	return YALM_OK;
}

// bf16 products of a few rows (M <= SK_MAX_T): the weight rows streamed once, in one or several K slices
template <bool GLU, class BMAP, class EPI>
static int stream_bf16(const PfForms &f, const uint16_t *A, int lda, int M, int K, const BMAP &bm, int N, const EPI &e,
                       float *part, size_t part_floats, hipStream_t st) {
	const StreamPlan p = plan_stream(M, N, K / 128, part_floats);
	const int np = (N + sk_cols(M) - 1) / sk_cols(M) * sk_cols(M);
	if (p.ks == 1)
		return launch_stream<false, GLU, true>(f, p, A, lda, M, K, K, bm, N, np, nullptr, e, st);
	TRY((launch_stream<false, GLU, true>(f, p, A, lda, M, K, K, bm, N, np, part, pf::NoEpi{}, st)));
	return launch_skinny_reduce<GLU>(part, p.ks, p.ks, np, M, np, e, st, sk_rows(M));
}

// The layer-list engine's door to the prefill GEMMs (seq.hip; device pointers, asynchronous
// on st): C [M][ldc] f32 = act(A [M][lda] bf16 . W [N][K]^T bf16 (+ bias[n])), act: E16StoreF32B. The same
// forms as the f16 prefill's: up to 64 rows the streamed split-K kernel (a 16-row product of [2048][2048] on the
// general kernel's 64 x 64 tiles is 32 workgroups, 60-100 us; so 8 + 4 us), else the large tiles, in K slices
// where plan_split says so (part: part_floats of scratch for the partials), else whole (an N that is no multiple
// of the tile takes a last tile that reaches past it). YALM_ERR_UNSUPPORTED (nothing launched) when the shape
// does not fit them: K % 64, N below one tile, rows not 16-byte aligned.
int pf_gemm_bf16(const uint16_t *A, int lda, int M, int K, const uint16_t *W, int N, float *C, int ldc,
                 const float *bias, int act, float *part, size_t part_floats, hipStream_t st) {
	static const PfForms f = pf_forms_default();
	if (M <= 0 || K % pf::BK != 0 || lda % 8 != 0 || ((size_t)A | (size_t)W) % 16 != 0)
		return YALM_ERR_UNSUPPORTED;
	const bool ragged = N % 128 != 0;
	const int bn = N < 128 ? 0 : pick_bn(f, PG_TEST, M, N, false, ragged);
	if (!bn)
		return YALM_ERR_UNSUPPORTED;
	pf::E16StoreF32B e;
	e.c = C;
	e.bias = bias;
	e.ldc = ldc;
	e.M = M;
	e.N = N;
	e.act = act;
	if (M <= SK_MAX_T && K % 128 == 0)
		return stream_bf16<false>(f, A, lda, M, K, pf::BRowsRagged{W, N}, N, e, part, part_floats, st);
	const SplitPlan s = plan_split(f, PG_TEST, M, N, K, 0, 0, false, part_floats, ragged);
	if (s.ks > 1) {
		TRY((launch_split<pf::BRowsRagged, true>(f, s, A, lda, M, K, K, pf::BRowsRagged{W, N}, s.n, 0, 0, part, st)));
		return launch_skinny_reduce<false>(part, s.ks, s.ks, s.n, M, s.n, e, st);
	}
	return launch_rows(f, bn, A, lda, M, K, K, pf::BRowsRagged{W, N}, (N + bn - 1) / bn * bn, e, st);
}

// The same door for a gated pair: C [M][ldc] f32 = act(A Wg^T) (.) (A Wu^T) over `hidden` units
// (mode / limit: E16GluB), the two matrices' rows interleaved per wave as in the f16 prefill.
int pf_gemm_glu_bf16(const uint16_t *A, int lda, int M, int K, const uint16_t *Wg, const uint16_t *Wu, int hidden,
                     float *C, int ldc, int mode, float limit, float *part, size_t part_floats, hipStream_t st) {
	static const PfForms f = pf_forms_default();
	if (M <= 0 || K % pf::BK != 0 || lda % 8 != 0 || ((size_t)A | (size_t)Wg | (size_t)Wu) % 16 != 0)
		return YALM_ERR_UNSUPPORTED;
	const int bn = pick_bn(f, PG_GLU, M, 2 * hidden, true);
	pf::E16GluB e;
	e.c = C;
	e.ldc = ldc;
	e.M = M;
	e.mode = mode;
	e.limit = limit;
	pf::BRowsGlu<64> bm{Wg, Wu};
	const int N = 2 * hidden;
	if (!bn)
		return YALM_ERR_UNSUPPORTED;
	if (M <= SK_MAX_T && K % 128 == 0 && N % sk_cols(M) == 0)
		return stream_bf16<true>(f, A, lda, M, K, bm, N, e, part, part_floats, st);
	const SplitPlan s = plan_split(f, PG_GLU, M, N, K, 0, 0, true, part_floats);
	if (s.ks > 1) {
		TRY((launch_split<pf::BRowsGlu<64>, true>(f, s, A, lda, M, K, K, bm, N, 0, 0, part, st)));
		return launch_skinny_reduce<true>(part, s.ks, s.ks, N, M, N, e, st);
	}
	if (bn == 256)
		return launch_g16_t<pf::E16GluB, pf::BRowsGlu<64>, 256, 2>(f, A, lda, M, K, K, bm, 2 * hidden, e, st);
	if (bn == 128)
		return launch_g16_t<pf::E16GluB, pf::BRowsGlu<64>, 128, 4>(f, A, lda, M, K, K, bm, 2 * hidden, e, st);
	return YALM_ERR_UNSUPPORTED;
}

// Products of groups of rows (routed experts): result row r of group g's list is A row r / a_div against the group's
// matrices, w_bs elements after the group's before it. `rows`: an upper bound of the lists' entries together.
// Width 256 or 128 by the time the expected tiles take (a group's last row tile half full), as plan_split counts it.
template <class EPI, class BMAP256, class BMAP128>
static int launch_groups(const uint16_t *A, int lda, int rows, int K, const BMAP256 &b256, const BMAP128 &b128, int N,
                         bool whole256, const EPI &epi, const pf::GrpRows &g, hipStream_t st) {
	const int ncu = (int)device_cu_count(), tm = rows / pf::G_BM + (g.n + 1) / 2;
	auto cost = [&](int w, int bn) {
		return (float)((tm * ((N + bn - 1) / bn) + ncu - 1) / ncu) * (K / pf::BK * T8P_KT[w] + T8P_TILE + T8P_EPI);
	};
	auto go = [&](auto kern, const auto &bm, size_t lds, int n, bool &attr) {
		if (!attr) {
			HIPCHK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
			attr = true;
		}
		hipLaunchKernelGGL(kern, dim3(ncu), dim3(pf::G_THREADS), lds, st, A, lda, 0, K, K, bm, n, epi, 0, n, K, 1 << 24, g);
		HIPCHK(hipGetLastError());
		return (int)YALM_OK;
	};
	static bool a256 = false, a128 = false;
	if (whole256 && cost(2, 256) <= cost(0, 128))
		return go(pf::gemm8p_kernel<EPI, BMAP256, 2, 2, pf::GrpRows>, b256, pf::gemm8p_lds<2, 2>(), (N + 255) / 256 * 256, a256);
	return go(pf::gemm8p_kernel<EPI, BMAP128, 1, 1, pf::GrpRows>, b128, pf::gemm8p_lds<1, 1>(), (N + 127) / 128 * 128, a128);
}
static bool groups_ok(const uint16_t *A, int lda, int rows, int K, const void *W, const void *W2, const pf::GrpRows &g) {
	return rows > 0 && K % pf::BK == 0 && lda % 8 == 0 && ((size_t)A | (size_t)W | (size_t)W2) % 16 == 0 && g.w_bs % 8 == 0 &&
	       g.n >= 1 && g.n <= 64 && (size_t)rows * lda < (size_t)1 << 32;
}
// The gated pair of the groups: C [rows][ldc] bf16 (mode / limit: E16GluB)
int pf_groups_glu_bf16(const uint16_t *A, int lda, int rows, int K, const uint16_t *Wg, const uint16_t *Wu, int hidden,
                       size_t w_bs, uint16_t *C, int ldc, int mode, float limit, const int *lists, int lists_bs,
                       const int *counts, int n, int a_div, hipStream_t st) {
	const pf::GrpRows g{lists, counts, n, lists_bs, a_div, w_bs};
	if (!groups_ok(A, lda, rows, K, Wg, Wu, g) || hidden % 64 != 0)
		return YALM_ERR_UNSUPPORTED;
	pf::E16GluBT<true> e;
	e.c = C;
	e.ldc = ldc;
	e.mode = mode;
	e.limit = limit;
	return launch_groups(A, lda, rows, K, pf::BRowsGlu<64>{Wg, Wu}, pf::BRowsGlu<32>{Wg, Wu}, 2 * hidden, hidden % 128 == 0, e, g, st);
}
// ... one matrix each, N rows: C [rows][ldc] f32
int pf_groups_bf16(const uint16_t *A, int lda, int rows, int K, const uint16_t *W, int N, size_t w_bs, float *C, int ldc,
                   const int *lists, int lists_bs, const int *counts, int n, int a_div, hipStream_t st) {
	const pf::GrpRows g{lists, counts, n, lists_bs, a_div, w_bs};
	if (!groups_ok(A, lda, rows, K, W, W, g))
		return YALM_ERR_UNSUPPORTED;
	pf::E16StoreRows e;
	e.c = C;
	e.ldc = ldc;
	e.N = N;
	return launch_groups(A, lda, rows, K, pf::BRowsRagged{W, N}, pf::BRowsRagged{W, N}, N, true, e, g, st);
}

extern "C" int yalm_gemm_f16(float *c, const uint16_t *a, const uint16_t *w, int M, int N, int K) {
	ARGCHK(c && a && w && M > 0 && N > 0 && K > 0, "yalm_gemm_f16: bad argument");
	ARGCHK(N % pf::BN == 0 && K % pf::BK == 0, "yalm_gemm_f16: N % 128 and K % 64 must be 0");
	HostDev da, dw, dc;
	TRY(hd(da, a, (size_t)M * K * 2));
	TRY(hd(dw, w, (size_t)N * K * 2));
	TRY(hd(dc, nullptr, (size_t)M * N * 4));
	pf::E16StoreF32 e16;
	e16.c = (float *)dc.p;
	e16.ldc = N;
	e16.M = M;
	const PfForms f = g_test_forms; // a test hook: the forms set by yalm_set_prefill_forms(NULL, ...)
	const size_t cap = (size_t)32 << 20; // as a decoder's (ensure_bufs)
	const SplitPlan s = plan_split(f, PG_TEST, M, N, K, 0, 0, false, cap);
	HostDev dp;
	if (s.ks > 1) { // K slices, summed by the reduce kernel the prefill uses
		const uint16_t *wp = (const uint16_t *)dw.p;
		TRY(hd(dp, nullptr, (size_t)s.ks * ((M + 15) / 16 * 16) * N * 4));
		TRY(launch_split(f, s, (const uint16_t *)da.p, K, M, K, K, pf::BRowsPlain{{{wp, wp, wp}, {N, N, N}}}, N, 0, 0,
		                 (float *)dp.p, nullptr));
		TRY(launch_skinny_reduce<false>((const float *)dp.p, s.ks, s.ks, N, M, N, e16, nullptr));
	} else {
		TRY(launch_plain(f, pick_bn(f, PG_TEST, M, N, false), (const uint16_t *)da.p, K, M, K, K, one(dw.p, N), N, e16,
		                 nullptr));
	}
	HIPCHK(hipDeviceSynchronize());
	HIPCHK(hipMemcpy(c, dc.p, (size_t)M * N * 4, hipMemcpyDeviceToHost));
	return YALM_OK;
}

extern "C" int yalm_attn_prefill(uint16_t *o, const uint16_t *q, const uint16_t *kc, const uint16_t *vc, int T,
                                 int pos0, int n_heads, int n_kv_heads, int head_dim) {
	ARGCHK(o && q && kc && vc && T > 0 && pos0 >= 0 && n_kv_heads > 0 && n_heads % n_kv_heads == 0,
	       "yalm_attn_prefill: bad argument");
	const size_t q_dim = (size_t)n_heads * head_dim, kv = (size_t)(pos0 + T) * n_kv_heads * head_dim;
	HostDev dq, dk, dv, dout;
	TRY(hd(dq, q, T * q_dim * 2));
	TRY(hd(dk, kc, kv * 2));
	TRY(hd(dv, vc, kv * 2));
	TRY(hd(dout, nullptr, T * q_dim * 2));
	TRY(launch_attn_prefill((const uint16_t *)dq.p, (const uint16_t *)dk.p, (const uint16_t *)dv.p, T, pos0, n_heads,
	                        n_kv_heads, head_dim, (uint16_t *)dout.p, nullptr));
	HIPCHK(hipDeviceSynchronize());
	HIPCHK(hipMemcpy(o, dout.p, T * q_dim * 2, hipMemcpyDeviceToHost));
	return YALM_OK;
}
