// gctf_fft.hpp -- LDS-resident complex FFTs for gfx950.
//
// Power-of-two lengths use a Stockham autosort (radix 8, last pass radix 2
// or 4) whose butterflies live in registers; one workgroup-wide barrier
// separates the LDS reads of a pass from its writes, so one LDS buffer of N
// complex values suffices.  Lengths 2^a 3^b 5^c run the same Stockham passes
// with further butterflies up to radix 12 (fft_mixed).  Other lengths
// run on a power-of-two grid at least twice as fine, reached by an eight-point
// interpolation (itp_fwd, itp_inv).  All are unnormalised; the forward
// transform uses exp(-2 pi i k n / N).
//
// LDS layout: logical element i lives at physical index pidx(i) = i + i/8.
// The Stockham writes of the early passes stride by the radix (8 complex);
// the odd multiplier 9 spreads those strides over all banks.  A buffer of N
// logical elements therefore needs fft_lds_len(N) = N + N/8 entries.
//
// Twiddles: one load w = exp(-2 pi i k S / N) per butterfly from a table
// computed on the host in double; the powers w^2 .. w^(R-1) are formed by
// complex products of depth <= 3.
//
// All code here is compiled with -ffp-contract=off; fused multiply-adds
// are written out with fmaf where they are wanted.
#pragma once
#include <hip/hip_runtime.h>

namespace gctf {

__host__ __device__ constexpr int fft_lds_len(int n) { return n + n / 8; }
__device__ __forceinline__ int pidx(int i) { return i + (i >> 3); }

__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
	return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.x, b.y, a.y * b.x));
}

// a * conj(b)
__device__ __forceinline__ float2 cmulc(float2 a, float2 b)
{
	return make_float2(fmaf(a.x, b.x, a.y * b.y), fmaf(a.y, b.x, -(a.x * b.y)));
}

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

// multiply by -i (forward) or +i (inverse)
template <bool INV>
__device__ __forceinline__ float2 mul_wi(float2 a)
{
	return INV ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

template <int R, bool INV>
__device__ __forceinline__ void dft_small(float2* u);

template <>
__device__ __forceinline__ void dft_small<2, false>(float2* u)
{
	float2 a = u[0], b = u[1];
	u[0] = cadd(a, b); u[1] = csub(a, b);
}
template <>
__device__ __forceinline__ void dft_small<2, true>(float2* u)
{
	float2 a = u[0], b = u[1];
	u[0] = cadd(a, b); u[1] = csub(a, b);
}

template <bool INV>
__device__ __forceinline__ void dft4(float2& a0, float2& a1, float2& a2, float2& a3)
{
	float2 t0 = cadd(a0, a2), t1 = csub(a0, a2);
	float2 t2 = cadd(a1, a3), t3 = mul_wi<INV>(csub(a1, a3));
	a0 = cadd(t0, t2); a2 = csub(t0, t2);
	a1 = cadd(t1, t3); a3 = csub(t1, t3);
}

template <>
__device__ __forceinline__ void dft_small<4, false>(float2* u) { dft4<false>(u[0], u[1], u[2], u[3]); }
template <>
__device__ __forceinline__ void dft_small<4, true>(float2* u) { dft4<true>(u[0], u[1], u[2], u[3]); }

template <bool INV>
__device__ __forceinline__ void dft8(float2* u)
{
	const float c = 0.70710678118654752f;
	float2 e0 = u[0], e1 = u[2], e2 = u[4], e3 = u[6];
	float2 o0 = u[1], o1 = u[3], o2 = u[5], o3 = u[7];
	dft4<INV>(e0, e1, e2, e3);
	dft4<INV>(o0, o1, o2, o3);
	// o_k *= W8^k
	float2 w1, w3;
	if (INV) {
		w1 = make_float2(c * (o1.x - o1.y), c * (o1.x + o1.y));
		w3 = make_float2(-c * (o3.x + o3.y), c * (o3.x - o3.y));
	} else {
		w1 = make_float2(c * (o1.x + o1.y), c * (o1.y - o1.x));
		w3 = make_float2(c * (o3.y - o3.x), -c * (o3.x + o3.y));
	}
	float2 w2 = mul_wi<INV>(o2);
	u[0] = cadd(e0, o0); u[4] = csub(e0, o0);
	u[1] = cadd(e1, w1); u[5] = csub(e1, w1);
	u[2] = cadd(e2, w2); u[6] = csub(e2, w2);
	u[3] = cadd(e3, w3); u[7] = csub(e3, w3);
}

template <>
__device__ __forceinline__ void dft_small<8, false>(float2* u) { dft8<false>(u); }
template <>
__device__ __forceinline__ void dft_small<8, true>(float2* u) { dft8<true>(u); }

// u1 (+-) i s u2 parts of the radix-3 and radix-5 butterflies: y = a + mul_wi(b)
// is a - i b forward, a + i b inverse.
template <bool INV>
__device__ __forceinline__ void dft3(float2* u)
{
	const float s3 = 0.86602540378443864676f;     // sin(2 pi / 3)
	const float2 t1 = cadd(u[1], u[2]);
	const float2 t2 = make_float2(fmaf(-0.5f, t1.x, u[0].x), fmaf(-0.5f, t1.y, u[0].y));
	const float2 d = mul_wi<INV>(make_float2(s3 * (u[1].x - u[2].x), s3 * (u[1].y - u[2].y)));
	u[0] = cadd(u[0], t1);
	u[1] = cadd(t2, d);
	u[2] = csub(t2, d);
}

template <bool INV>
__device__ __forceinline__ void dft5(float2* u)
{
	const float c1 = 0.30901699437494742410f;     // cos(2 pi / 5)
	const float c2 = -0.80901699437494742410f;    // cos(4 pi / 5)
	const float s1 = 0.95105651629515357212f;     // sin(2 pi / 5)
	const float s2 = 0.58778525229247312917f;     // sin(4 pi / 5)
	const float2 a1 = cadd(u[1], u[4]), a2 = cadd(u[2], u[3]);
	const float2 b1 = csub(u[1], u[4]), b2 = csub(u[2], u[3]);
	const float2 p1 = make_float2(fmaf(c2, a2.x, fmaf(c1, a1.x, u[0].x)), fmaf(c2, a2.y, fmaf(c1, a1.y, u[0].y)));
	const float2 p2 = make_float2(fmaf(c1, a2.x, fmaf(c2, a1.x, u[0].x)), fmaf(c1, a2.y, fmaf(c2, a1.y, u[0].y)));
	const float2 q1 = mul_wi<INV>(make_float2(fmaf(s2, b2.x, s1 * b1.x), fmaf(s2, b2.y, s1 * b1.y)));
	const float2 q2 = mul_wi<INV>(make_float2(fmaf(-s1, b2.x, s2 * b1.x), fmaf(-s1, b2.y, s2 * b1.y)));
	u[0] = cadd(cadd(u[0], a1), a2);
	u[1] = cadd(p1, q1);
	u[4] = csub(p1, q1);
	u[2] = cadd(p2, q2);
	u[3] = csub(p2, q2);
}

template <>
__device__ __forceinline__ void dft_small<3, false>(float2* u) { dft3<false>(u); }
template <>
__device__ __forceinline__ void dft_small<3, true>(float2* u) { dft3<true>(u); }
template <>
__device__ __forceinline__ void dft_small<5, false>(float2* u) { dft5<false>(u); }
template <>
__device__ __forceinline__ void dft_small<5, true>(float2* u) { dft5<true>(u); }

// Composite radices: N = A B coprime (Good-Thomas, no twiddles): the inputs
// (B a + A b) mod N, the outputs (KA a + KB b) mod N with KA = 1 mod A, 0 mod
// B and KB the reverse.
template <int A, int B, int KA, int KB, bool INV>
__device__ __forceinline__ void dft_coprime(float2* u)
{
	constexpr int N = A * B;
	static_assert(KA % A == 1 && KA % B == 0 && KB % B == 1 && KB % A == 0, "residues");
	float2 v[A][B];
#pragma unroll
	for (int a = 0; a < A; ++a) {
#pragma unroll
		for (int b = 0; b < B; ++b) v[a][b] = u[(B * a + A * b) % N];
		dft_small<B, INV>(v[a]);
	}
#pragma unroll
	for (int b = 0; b < B; ++b) {
		float2 c[A];
#pragma unroll
		for (int a = 0; a < A; ++a) c[a] = v[a][b];
		dft_small<A, INV>(c);
#pragma unroll
		for (int a = 0; a < A; ++a) u[(KA * a + KB * b) % N] = c[a];
	}
}
template <> __device__ __forceinline__ void dft_small<6, false>(float2* u) { dft_coprime<2, 3, 3, 4, false>(u); }
template <> __device__ __forceinline__ void dft_small<6, true>(float2* u) { dft_coprime<2, 3, 3, 4, true>(u); }
template <> __device__ __forceinline__ void dft_small<10, false>(float2* u) { dft_coprime<2, 5, 5, 6, false>(u); }
template <> __device__ __forceinline__ void dft_small<10, true>(float2* u) { dft_coprime<2, 5, 5, 6, true>(u); }
template <> __device__ __forceinline__ void dft_small<12, false>(float2* u) { dft_coprime<4, 3, 9, 4, false>(u); }
template <> __device__ __forceinline__ void dft_small<12, true>(float2* u) { dft_coprime<4, 3, 9, 4, true>(u); }

// 9 = 3 x 3, twiddles exp(-+2 pi i a b / 9)
template <bool INV>
__device__ __forceinline__ void dft9(float2* u)
{
	const float2 w1 = make_float2(0.76604444311897803520f, INV ? 0.64278760968653932632f : -0.64278760968653932632f);
	const float2 w2 = make_float2(0.17364817766693034885f, INV ? 0.98480775301220805937f : -0.98480775301220805937f);
	const float2 w4 = make_float2(-0.93969262078590838405f, INV ? 0.34202014332566873304f : -0.34202014332566873304f);
	float2 v[3][3];
#pragma unroll
	for (int b = 0; b < 3; ++b) {
		v[b][0] = u[b]; v[b][1] = u[b + 3]; v[b][2] = u[b + 6];
		dft3<INV>(v[b]);
	}
	v[1][1] = cmul(v[1][1], w1); v[1][2] = cmul(v[1][2], w2);
	v[2][1] = cmul(v[2][1], w2); v[2][2] = cmul(v[2][2], w4);
#pragma unroll
	for (int a = 0; a < 3; ++a) {
		float2 c[3] = {v[0][a], v[1][a], v[2][a]};
		dft3<INV>(c);
		u[a] = c[0]; u[a + 3] = c[1]; u[a + 6] = c[2];
	}
}
template <> __device__ __forceinline__ void dft_small<9, false>(float2* u) { dft9<false>(u); }
template <> __device__ __forceinline__ void dft_small<9, true>(float2* u) { dft9<true>(u); }

// u[r] *= w^r for r = 1 .. R-1 (w already conjugated for the inverse).
template <int R>
__device__ __forceinline__ void twiddle_powers(float2* u, float2 w)
{
	float2 p[R];
	p[1] = w;
#pragma unroll
	for (int r = 2; r < R; ++r) {
		int hb = 1;
		while (hb * 2 <= r) hb *= 2;
		p[r] = (hb == r) ? cmul(p[r / 2], p[r / 2]) : cmul(p[hb], p[r - hb]);
	}
#pragma unroll
	for (int r = 1; r < R; ++r) u[r] = cmul(u[r], p[r]);
}

// Synchronisation of the NT threads that share one transform.  A transform
// of at most 64 threads belongs to a single wavefront: its LDS accesses
// execute in issue order, so a wavefront-scope fence (which keeps the
// compiler from moving LDS accesses across it and waits for the outstanding
// ones) replaces the workgroup barrier, and the other transforms of the
// workgroup run on.
template <int NT>
__device__ __forceinline__ void fft_sync()
{
	if constexpr (NT <= 64) {
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
	} else {
		__syncthreads();
	}
}

// Twiddle sources of the power-of-two passes.  Pass P (its L > 1) of
// butterfly b of thread j uses w = exp(-2 pi i k S / N) with k = j mod L,
// S = N / (L R).  TwTable loads it from the table where the pass needs it;
// TwRegs holds every pass's values in registers, loaded once (fft_tw_load)
// by a kernel that runs many transforms of one length with the same threads:
// the passes then wait for no memory, and a load issued before the
// transform (the next transform's input) stays in flight through it.
struct TwTable {
	const float2* __restrict__ tw;
	template <int N, int R, int L, int P>
	__device__ __forceinline__ float2 get(int, int j) const { return tw[(j & (L - 1)) * (N / (L * R))]; }
};

// Passes of the power-of-two Stockham transform of length N (radix 8, the
// last 2 or 4) and the largest butterfly count per thread of any of them.
__host__ __device__ constexpr int fft_npass(int n)
{
	int p = 0;
	for (int l = 1; l < n; l *= (n / l >= 8 ? 8 : n / l)) ++p;
	return p;
}
__host__ __device__ constexpr int fft_max_bpt(int n, int nt)
{
	int m = 1;
	for (int l = 1; l < n; l *= (n / l >= 8 ? 8 : n / l)) {
		const int t = n / (n / l >= 8 ? 8 : n / l);
		m = (t + nt - 1) / nt > m ? (t + nt - 1) / nt : m;
	}
	return m;
}

template <int N, int NT>
struct TwRegs {
	float2 v[fft_npass(N)][fft_max_bpt(N, NT)];
	template <int N2, int R, int L, int P>
	__device__ __forceinline__ float2 get(int b, int) const { return v[P][b]; }
};

template <int N, int L, int NT, int P>
__device__ __forceinline__ void fft_tw_load_run(TwRegs<N, NT>& w, const float2* __restrict__ tw, int tid)
{
	if constexpr (L < N) {
		constexpr int rem = N / L;
		constexpr int R = rem >= 8 ? 8 : rem;
		if constexpr (L > 1) {
			constexpr int T = N / R;
			constexpr int BPT = (T + NT - 1) / NT;
#pragma unroll
			for (int b = 0; b < BPT; ++b) {
				const int j = tid + b * NT;
				if (T % NT == 0 || j < T) w.v[P][b] = tw[(j & (L - 1)) * (N / (L * R))];
			}
		}
		fft_tw_load_run<N, L * R, NT, P + 1>(w, tw, tid);
	}
}

// The twiddles thread tid of fft_lds<N, NT, INV> uses, from the table tw.
template <int N, int NT>
__device__ __forceinline__ void fft_tw_load(TwRegs<N, NT>& w, const float2* __restrict__ tw, int tid)
{
	fft_tw_load_run<N, 1, NT, 0>(w, tw, tid);
}

// The LDS addresses of a butterfly's R elements i0 + r D.  With D a multiple of
// 8, or i0 a multiple of 8 and D = 1, R <= 8, the padding adds the same to every
// step: one base address and constant offsets, which the LDS instructions take
// as immediates, instead of a register and two instructions each.  Tile rows 69
// -> 61 VGPRs, 41 x 3838x3710 spectra 4333 -> 4295 us.  The passes with hooks
// (fft_run_io) keep the plain form: their columns took 2076 us per 32 x 4096^2
// with it and 2130 with this one.
template <int R, int D>
__device__ __forceinline__ void lds_read(float2* u, const float2* buf, int i0)
{
	if constexpr (D % 8 == 0) {
		const float2* p = buf + pidx(i0);
#pragma unroll
		for (int r = 0; r < R; ++r) u[r] = p[r * (D + D / 8)];
	} else {
#pragma unroll
		for (int r = 0; r < R; ++r) u[r] = buf[pidx(i0 + r * D)];
	}
}
// UNIT8: i0 is a multiple of 8 (and D is 1)
template <int R, int D, bool UNIT8 = false>
__device__ __forceinline__ void lds_write(float2* buf, int i0, const float2* u)
{
	if constexpr (D % 8 == 0 || (UNIT8 && D == 1 && R <= 8)) {
		float2* p = buf + pidx(i0);
#pragma unroll
		for (int r = 0; r < R; ++r) p[r * (D + D / 8)] = u[r];
	} else {
#pragma unroll
		for (int r = 0; r < R; ++r) buf[pidx(i0 + r * D)] = u[r];
	}
}

// One Stockham pass of radix R over N points; L = product of the radices of
// the previous passes; P its index.  NT threads (tid in [0, NT)) share the
// buffer.
template <int N, int R, int L, int P, int NT, bool INV, class TW>
__device__ __forceinline__ void fft_pass(float2* buf, const TW& twf, int tid)
{
	constexpr int T = N / R;
	constexpr int BPT = (T + NT - 1) / NT;
	float2 u[BPT][R];
#pragma unroll
	for (int b = 0; b < BPT; ++b) {
		const int j = tid + b * NT;
		if (T % NT == 0 || j < T) {
			lds_read<R, T>(u[b], buf, j);
			if constexpr (L > 1) {
				float2 w = twf.template get<N, R, L, P>(b, j);
				if (INV) w.y = -w.y;
				twiddle_powers<R>(u[b], w);
			}
			dft_small<R, INV>(u[b]);
		}
	}
	fft_sync<NT>();
#pragma unroll
	for (int b = 0; b < BPT; ++b) {
		const int j = tid + b * NT;
		if (T % NT == 0 || j < T) {
			const int k = j & (L - 1);
			const int base = (j - k) * R + k;
			lds_write<R, L, R == 8>(buf, base, u[b]);
		}
	}
	fft_sync<NT>();
}

template <int N, int L, int P, int NT, bool INV, class TW>
__device__ __forceinline__ void fft_run(float2* buf, const TW& twf, int tid)
{
	if constexpr (L < N) {
		constexpr int rem = N / L;
		constexpr int R = rem >= 8 ? 8 : rem;
		fft_pass<N, R, L, P, NT, INV>(buf, twf, tid);
		fft_run<N, L * R, P + 1, NT, INV>(buf, twf, tid);
	}
}

// The transform of N = 8 NT elements from registers to registers: thread tid
// holds elements x[i] = input tid + i NT and gets x[i] = output tid + i NT.
// Those are exactly the inputs of its first (radix-8) butterfly and the
// outputs of its last ones, so a transform makes one LDS round trip per pass
// boundary (two for 512 points) instead of one more at either end.  Same
// arithmetic as fft_lds.  buf may still be read by the NT threads' previous
// transform; its contents afterwards are not defined, and it may be reused
// after an fft_sync.
template <int N, int L, int P, int NT, bool INV, class TW>
__device__ __forceinline__ void fft_regs_run(float2* buf, const TW& twf, int tid, float2 (&x)[N / NT])
{
	constexpr int rem = N / L;
	constexpr int R = rem >= 8 ? 8 : rem;
	if constexpr (L * R < N) {
		fft_pass<N, R, L, P, NT, INV>(buf, twf, tid);
		fft_regs_run<N, L * R, P + 1, NT, INV>(buf, twf, tid, x);
	} else {
		constexpr int T = N / R, BPT = T / NT;
#pragma unroll
		for (int b = 0; b < BPT; ++b) {
			const int j = tid + b * NT;
			float2 u[R];
			lds_read<R, T>(u, buf, j);
			float2 w = twf.template get<N, R, L, P>(b, j);
			if (INV) w.y = -w.y;
			twiddle_powers<R>(u, w);
			dft_small<R, INV>(u);
#pragma unroll
			for (int r = 0; r < R; ++r) x[b + BPT * r] = u[r];
		}
	}
}

template <int N, int NT, bool INV, class TW>
__device__ __forceinline__ void fft_regs(float2* buf, const TW& twf, int tid, float2 (&x)[N / NT])
{
	static_assert(N == 8 * NT && N > 64, "one radix-8 butterfly per thread, and a pass after it");
	dft_small<8, INV>(x);
	fft_sync<NT>();
	lds_write<8, 1, true>(buf, 8 * tid, x);
	fft_sync<NT>();
	fft_regs_run<N, 8, 1, NT, INV>(buf, twf, tid, x);
}

// In-place power-of-two FFT of the N logical elements of buf (padded
// layout, fft_lds_len(N) entries) by NT threads.  With NT <= 64 the threads
// must be in one wavefront and only they synchronise (fft_sync); otherwise
// every thread of the workgroup must call it.  The data must be in buf and
// visible (fft_sync<NT> or a barrier) before the call; results are visible
// to the NT threads after.
template <int N, int NT, bool INV>
__device__ __forceinline__ void fft_lds(float2* buf, const float2* __restrict__ tw, int tid)
{
	fft_run<N, 1, 0, NT, INV>(buf, TwTable{tw}, tid);
}

// ---- compile-time transform with input and output hooks -----------------
// fft_lds_io runs the same passes as fft_lds, but the first pass takes its
// inputs from ld(i) (logical input index i) instead of buf, and the last
// pass hands its outputs to st(i, v) instead of storing v at buf[pidx(i)].
// ld may read buf: every read of a pass precedes its writes.  st may write
// anywhere in buf: the last pass's reads are over when it is called, and an
// fft_sync follows.  Loading and pointwise work before and after a transform
// then cost no LDS round trip and no barrier of their own.

// The plain output: buf itself.
struct LdsOut {
	float2* buf;
	__device__ __forceinline__ void operator()(int i, float2 v) const { buf[pidx(i)] = v; }
};

// A pass's twiddles are loaded before the barrier that precedes it, so that
// their latency (L2, several hundred cycles) overlaps the stores and the wait.
template <int N, int L>
__host__ __device__ constexpr int fft_radix() { return N / L >= 8 ? 8 : N / L; }

template <int N, int L, int NT>
__device__ __forceinline__ void fft_tw_fetch(float2* w, const float2* __restrict__ tw, int tid)
{
	constexpr int R = fft_radix<N, L>(), T = N / R, BPT = (T + NT - 1) / NT;
#pragma unroll
	for (int b = 0; b < BPT; ++b) {
		const int j = tid + b * NT;
		if (T % NT == 0 || j < T) w[b] = tw[(j & (L - 1)) * (N / (L * R))];
	}
}

template <int N, int L, int NT, bool INV, class Ld, class St>
__device__ __forceinline__ void fft_run_io(float2* buf, const float2* __restrict__ tw, int tid,
	const Ld& ld, const St& st, const float2* w)
{
	if constexpr (L < N) {
		constexpr int R = fft_radix<N, L>(), T = N / R;
		constexpr int BPT = (T + NT - 1) / NT;
		float2 u[BPT][R];
#pragma unroll
		for (int b = 0; b < BPT; ++b) {
			const int j = tid + b * NT;
			if (T % NT == 0 || j < T) {
#pragma unroll
				for (int r = 0; r < R; ++r) {
					if constexpr (L == 1) u[b][r] = ld(j + r * T);
					else u[b][r] = buf[pidx(j + r * T)];
				}
				if constexpr (L > 1) {
					float2 wb = w[b];
					if (INV) wb.y = -wb.y;
					twiddle_powers<R>(u[b], wb);
				}
				dft_small<R, INV>(u[b]);
			}
		}
		constexpr int L2 = L * R;
		float2 wn[fft_max_bpt(N, NT)];
		if constexpr (L2 < N) fft_tw_fetch<N, L2, NT>(wn, tw, tid);
		fft_sync<NT>();
#pragma unroll
		for (int b = 0; b < BPT; ++b) {
			const int j = tid + b * NT;
			if (T % NT == 0 || j < T) {
				const int k = j & (L - 1);
				const int base = (j - k) * R + k;
#pragma unroll
				for (int r = 0; r < R; ++r) {
					if constexpr (L2 == N) st(base + r * L, u[b][r]);
					else buf[pidx(base + r * L)] = u[b][r];
				}
			}
		}
		fft_sync<NT>();
		fft_run_io<N, L2, NT, INV>(buf, tw, tid, ld, st, wn);
	}
}

// Same contract as fft_lds, except that the first pass reads ld(i) and the
// last pass writes through st.  N >= 16 (the first pass is not the last).
template <int N, int NT, bool INV, class Ld, class St>
__device__ __forceinline__ void fft_lds_io(float2* buf, const float2* __restrict__ tw, int tid,
	const Ld& ld, const St& st)
{
	static_assert(N >= 16, "the first and last passes must differ");
	fft_run_io<N, 1, NT, INV>(buf, tw, tid, ld, st, nullptr);
}

// ---- runtime-length power-of-two FFT (lengths up to MAXN) ----------------
template <int R, int NT, int MAXN, bool INV>
__device__ __forceinline__ void fft_pass_rt(float2* buf, const float2* __restrict__ tw, int tid,
	int L, int T, int S)
{
	constexpr int BPT = (MAXN / R + NT - 1) / NT;
	float2 u[BPT][R];
#pragma unroll
	for (int b = 0; b < BPT; ++b) {
		const int j = tid + b * NT;
		if (j < T) {
#pragma unroll
			for (int r = 0; r < R; ++r) u[b][r] = buf[pidx(j + r * T)];
			if (L > 1) {
				const int k = j & (L - 1);
				float2 w = tw[k * S];
				if (INV) w.y = -w.y;
				twiddle_powers<R>(u[b], w);
			}
			dft_small<R, INV>(u[b]);
		}
	}
	__syncthreads();
#pragma unroll
	for (int b = 0; b < BPT; ++b) {
		const int j = tid + b * NT;
		if (j < T) {
			const int k = j & (L - 1);
			const int base = (j - k) * R + k;
#pragma unroll
			for (int r = 0; r < R; ++r) buf[pidx(base + r * L)] = u[b][r];
		}
	}
	__syncthreads();
}

// In-place power-of-two FFT of runtime length n <= MAXN; same contract as
// fft_lds.  The lengths MAXN and MAXN/2 run the compile-time transform (the
// same arithmetic, with its LDS addresses computed once per thread instead
// of once per pass); other lengths loop over runtime passes.
template <int NT, int MAXN, bool INV>
__device__ __forceinline__ void fft_lds_rt(float2* buf, int n, const float2* __restrict__ tw, int tid)
{
	if (n == MAXN) {
		fft_lds<MAXN, NT, INV>(buf, tw, tid);
		return;
	}
	if (n == MAXN / 2) {
		fft_lds<MAXN / 2, NT, INV>(buf, tw, tid);
		return;
	}
	int L = 1;
	while (L < n) {
		const int rem = n / L;
		if (rem >= 8) {
			fft_pass_rt<8, NT, MAXN, INV>(buf, tw, tid, L, n / 8, n / (L * 8));
			L *= 8;
		} else if (rem == 4) {
			fft_pass_rt<4, NT, MAXN, INV>(buf, tw, tid, L, n / 4, 1);
			L *= 4;
		} else {
			fft_pass_rt<2, NT, MAXN, INV>(buf, tw, tid, L, n / 2, 1);
			L *= 2;
		}
	}
}

// A 1D transform of arbitrary length n in LDS, as planned on the host.
struct Fft1dPlan {
	int n;                   // transform length
	int m;                   // working length: n for powers of two and for lengths 2^a 3^b 5^c,
	                         // else the points of the fine grid, the kernel's MAXN
	const float2* tw;        // twiddles of the passes: n points, or m / 2 points on the fine grid
	int nrad;                // mixed-radix passes (lengths 2^a 3^b 5^c that are not powers of two), else 0
	unsigned char rad[20];   // their radices, in pass order
	// lengths on the fine grid (else null); S = 2 when n is even, else 1
	const float2* mode;      // [2][n/2 + 1]: the modes' factors on the grid's even and odd points
	const float4* w8;        // [n/S][2]: the 8 weights of output t around point p0[t] (inverse)
	const int* p0;           // [n/S]
	const float4* w4;        // [2][m/2/S]: the 4 weights of fine point 2 i + b from input q0[b][i] on (forward)
	const int* q0;           // [2][m/2/S]
};

// ---- mixed-radix FFT (lengths 2^a 3^b 5^c) --------------------------------
// The Stockham pass of radix R after passes of product L, for any radices:
// butterfly j (T = n / R of them) reads j + r T, multiplies element r by
// w^r with w = exp(-+2 pi i k S / n), k = j mod L, S = n / (L R), and
// writes (j - k) R + k + r L.
//
// What bounds it is the chain of a pass (LDS, twiddle load, barrier), so the
// radices are as large as fit in registers (mixed_radices): 5760 = 8 8 10 9
// in 4 passes instead of 8 8 2 3 3 5 in 6.  A pass enters with the barrier
// that follows the last one's writes still to come and loads its twiddles
// before it.  Where T (or L) is a multiple of 8, as after a first radix of 8,
// the padded addresses of a butterfly's reads (writes) are equally spaced.
template <int R, int NT, int MAXN, bool INV>
__device__ __forceinline__ void fft_pass_mx(float2* buf, const float2* __restrict__ tw, int tid,
	int L, int T, int S)
{
	constexpr int BPT = (MAXN / R + NT - 1) / NT;
	// q = j / L: (j + 1/2) / L is at least 1 / (2 L) from an integer, and its
	// rounding error below 2^-23 j / L, less for j < 2^14
	const float rl = 1.0f / (float)L;
	float2 u[BPT][R], w[BPT];
	int kk[BPT];
#pragma unroll
	for (int b = 0; b < BPT; ++b) {
		const int j = tid + b * NT;
		kk[b] = j - (int)(((float)j + 0.5f) * rl) * L;
		if (j < T) w[b] = tw[kk[b] * S];
	}
	__syncthreads();
	const bool even_reads = (T & 7) == 0;
#pragma unroll
	for (int b = 0; b < BPT; ++b) {
		const int j = tid + b * NT;
		if (j < T) {
			if (even_reads) {
				const float2* p = buf + pidx(j);
				const int st = T + (T >> 3);
#pragma unroll
				for (int r = 0; r < R; ++r) u[b][r] = p[r * st];
			} else {
#pragma unroll
				for (int r = 0; r < R; ++r) u[b][r] = buf[pidx(j + r * T)];
			}
			if (L > 1) {
				float2 wb = w[b];
				if (INV) wb.y = -wb.y;
				twiddle_powers<R>(u[b], wb);
			}
			dft_small<R, INV>(u[b]);
		}
	}
	__syncthreads();
	const bool even_writes = (L & 7) == 0;
#pragma unroll
	for (int b = 0; b < BPT; ++b) {
		const int j = tid + b * NT;
		if (j < T) {
			const int base = (j - kk[b]) * R + kk[b];
			if (even_writes) {
				float2* p = buf + pidx(base);
				const int st = L + (L >> 3);
#pragma unroll
				for (int r = 0; r < R; ++r) p[r * st] = u[b][r];
			} else {
#pragma unroll
				for (int r = 0; r < R; ++r) buf[pidx(base + r * L)] = u[b][r];
			}
		}
	}
}

// The passes of a mixed-radix plan (n <= MAXN) from pass i on; the data is in
// buf, not necessarily visible yet; results are visible after.
template <int NT, int MAXN, bool INV>
__device__ __forceinline__ void fft_lds_mixed(float2* buf, const Fft1dPlan& p, int tid, int i, int L)
{
	for (; i < p.nrad; ++i) {
		const int R = p.rad[i];
		const int T = p.n / R, S = p.n / (L * R);
		if (R == 8) fft_pass_mx<8, NT, MAXN, INV>(buf, p.tw, tid, L, T, S);
		else if (R == 10) fft_pass_mx<10, NT, MAXN, INV>(buf, p.tw, tid, L, T, S);
		else if (R == 9) fft_pass_mx<9, NT, MAXN, INV>(buf, p.tw, tid, L, T, S);
		else if (R == 12) fft_pass_mx<12, NT, MAXN, INV>(buf, p.tw, tid, L, T, S);
		else if (R == 6) fft_pass_mx<6, NT, MAXN, INV>(buf, p.tw, tid, L, T, S);
		else if (R == 4) fft_pass_mx<4, NT, MAXN, INV>(buf, p.tw, tid, L, T, S);
		else if (R == 2) fft_pass_mx<2, NT, MAXN, INV>(buf, p.tw, tid, L, T, S);
		else if (R == 3) fft_pass_mx<3, NT, MAXN, INV>(buf, p.tw, tid, L, T, S);
		else fft_pass_mx<5, NT, MAXN, INV>(buf, p.tw, tid, L, T, S);
		L *= R;
	}
	__syncthreads();
}

// The transform of src(i), i in [0, n), by a mixed-radix plan, result in
// logical buf[0..n).  src may read buf.  A first radix of 8 takes its inputs
// straight from src.
template <int NT, int MAXN, bool INV, class Src>
__device__ __forceinline__ void fft_mixed(float2* buf, const Fft1dPlan& p, int tid, const Src& src)
{
	if (p.rad[0] == 8) {
		constexpr int BPT = (MAXN / 8 + NT - 1) / NT;
		const int T = p.n / 8;
		float2 u[BPT][8];
#pragma unroll
		for (int b = 0; b < BPT; ++b) {
			const int j = tid + b * NT;
			if (j < T) {
#pragma unroll
				for (int r = 0; r < 8; ++r) u[b][r] = src(j + r * T);
				dft8<INV>(u[b]);
			}
		}
		__syncthreads();
#pragma unroll
		for (int b = 0; b < BPT; ++b) {
			const int j = tid + b * NT;
			if (j < T) {
#pragma unroll
				for (int r = 0; r < 8; ++r) buf[9 * j + r] = u[b][r];     // pidx(8 j + r)
			}
		}
		fft_lds_mixed<NT, MAXN, INV>(buf, p, tid, 1, 8);
		return;
	}
	constexpr int PER = (MAXN + NT - 1) / NT;
	float2 v[PER];
#pragma unroll
	for (int b = 0; b < PER; ++b) {
		const int i = tid + b * NT;
		if (i < p.n) v[b] = src(i);
	}
	__syncthreads();
#pragma unroll
	for (int b = 0; b < PER; ++b) {
		const int i = tid + b * NT;
		if (i < p.n) buf[pidx(i)] = v[b];
	}
	fft_lds_mixed<NT, MAXN, INV>(buf, p, tid, 0, 1);
}

// ---- other lengths: a transform on a finer power-of-two grid ---------------
// The DFT of any length n on a grid of m = 2 P points, P >= n a power of two,
// by a band-limited interpolation kernel phi (Kaiser-Bessel, 8 fine points
// wide, Fourier transform phi^):
//   inverse:  y[t] = sum_k Y[k] exp(2 pi i k t / n), |k| <= n/2, is the
//     trigonometric polynomial of the modes at t m / n on the fine grid.  With
//     g[l] = sum_k (Y[k] / phi^(k/m)) exp(2 pi i k l / m),
//     y[t] = sum over 8 points l of phi(t m/n - l) g[l].  The even and the odd
//     points of g are one P-point inverse transform each, the odd one of the
//     modes turned by exp(pi i k / P): no zero padding is transformed.
//   forward: the adjoint.  f[l] = sum of phi(l - j m/n) x[j], at most 4 inputs
//     per fine point; X[k] = (E[k] + exp(-pi i k / P) O[k]) / phi^(k/m) with
//     E, O the P-point transforms of f's even and odd points.
// At oversampling m/n >= 2 the kernel's aliasing is below 6e-8 of the result
// (2e-8 at m/n = 2.4), under the FP32 rounding of the transforms.
//
// Why: Bluestein's convolution needs two m-point transforms of which half is
// padding; this needs two P-point ones and 8 (4) multiply-adds per point.
// Each half of the workgroup runs one of the two, in its half of buf; every
// sync spans the workgroup (NT/2 > 64).
constexpr int kItpHalo = 4;   // entries kept on either side of a periodic LDS array

// For n even the outputs t and t + n/2 of the inverse have the same weights,
// half the grid apart.  TOBUF: out may write buf (it is called after every
// read of the grid).
template <int NT, int MAXN, bool TOBUF, class Src, class Out>
__device__ __forceinline__ void itp_inv(float2* buf, const Fft1dPlan& p, int tid, const Src& src, const Out& out)
{
	constexpr int P = MAXN / 2, HT = NT / 2, RL = fft_lds_len(P), H = kItpHalo;
	static_assert(HT > 64, "the halves' barriers must span the workgroup");
	static_assert(P + 2 * H <= RL, "the halo fits a half of the buffer");
	const int g = tid / HT, lt = tid - g * HT;
	float2* hb = buf + g * RL;
	const int n = p.n, kmax = n / 2, kmin = -((n - 1) / 2);
	const float2* mode = p.mode + g * (kmax + 1);
	auto ld = [&](int i) -> float2 {
		const int k = i < P / 2 ? i : i - P;
		const bool in = k >= kmin && k <= kmax;
		const int kc = min(max(k, kmin), kmax);
		const float2 f = mode[kc < 0 ? -kc : kc];
		const float2 v = src(kc);
		const float2 r = kc < 0 ? cmulc(v, f) : cmul(v, f);
		return in ? r : make_float2(0.f, 0.f);
	};
	// the grid's half, linear with its periodic halo
	auto st = [&](int i, float2 v) {
		hb[i + H] = v;
		if (i < H) hb[i + H + P] = v;
		if (i >= P - H) hb[i + H - P] = v;
	};
	fft_lds_io<P, HT, true>(hb, p.tw, lt, ld, st);
	auto at = [&](const float4& wa, const float4& wb, int l0, int shift) -> float2 {
		// points l0 .. l0 + 7: the halves alternate, starting with l0's
		const int e = l0 >> 1, odd = l0 & 1;
		const float2* ga = buf + (odd ? RL : 0) + e + H + shift;
		const float2* gb = buf + (odd ? 0 : RL) + e + odd + H + shift;
		float2 s = make_float2(wa.x * ga[0].x, wa.x * ga[0].y);
		s.x = fmaf(wa.y, gb[0].x, s.x); s.y = fmaf(wa.y, gb[0].y, s.y);
		s.x = fmaf(wa.z, ga[1].x, s.x); s.y = fmaf(wa.z, ga[1].y, s.y);
		s.x = fmaf(wa.w, gb[1].x, s.x); s.y = fmaf(wa.w, gb[1].y, s.y);
		s.x = fmaf(wb.x, ga[2].x, s.x); s.y = fmaf(wb.x, ga[2].y, s.y);
		s.x = fmaf(wb.y, gb[2].x, s.x); s.y = fmaf(wb.y, gb[2].y, s.y);
		s.x = fmaf(wb.z, ga[3].x, s.x); s.y = fmaf(wb.z, ga[3].y, s.y);
		s.x = fmaf(wb.w, gb[3].x, s.x); s.y = fmaf(wb.w, gb[3].y, s.y);
		return s;
	};
	// PER outputs per thread at most; with n even two of them per weight set
	constexpr int PER = (P + NT - 1) / NT;
	static_assert(PER % 2 == 0, "outputs t and t + n/2 in pairs");
	float2 v[PER];
	if (n % 2 == 0) {
#pragma unroll
		for (int b = 0; b < PER / 2; ++b) {
			const int t = tid + b * NT;
			if (t < n / 2) {
				const float4 wa = p.w8[2 * t], wb = p.w8[2 * t + 1];
				const int l0 = p.p0[t];
				v[2 * b] = at(wa, wb, l0, 0);
				v[2 * b + 1] = at(wa, wb, l0, P / 2);
				if constexpr (!TOBUF) {
					out(t, v[2 * b]);
					out(t + n / 2, v[2 * b + 1]);
				}
			}
		}
		if constexpr (TOBUF) {
			__syncthreads();
#pragma unroll
			for (int b = 0; b < PER / 2; ++b) {
				const int t = tid + b * NT;
				if (t < n / 2) {
					out(t, v[2 * b]);
					out(t + n / 2, v[2 * b + 1]);
				}
			}
		}
	} else {
#pragma unroll
		for (int b = 0; b < PER; ++b) {
			const int t = tid + b * NT;
			if (t < n) {
				v[b] = at(p.w8[2 * t], p.w8[2 * t + 1], p.p0[t], 0);
				if constexpr (!TOBUF) out(t, v[b]);
			}
		}
		if constexpr (TOBUF) {
			__syncthreads();
#pragma unroll
			for (int b = 0; b < PER; ++b) {
				const int t = tid + b * NT;
				if (t < n) out(t, v[b]);
			}
		}
	}
}

// The forward transform; result in logical buf[0..n) (visible to the
// workgroup).
template <int NT, int MAXN, class Src>
__device__ __forceinline__ void itp_fwd(float2* buf, const Fft1dPlan& p, int tid, const Src& src)
{
	constexpr int P = MAXN / 2, HT = NT / 2, RL = fft_lds_len(P), H = kItpHalo;
	static_assert(HT > 64, "the halves' barriers must span the workgroup");
	const int g = tid / HT, lt = tid - g * HT;
	float2* hb = buf + g * RL;
	const int n = p.n;
	constexpr int PER = (P + NT - 1) / NT;
	{
		float2 v[PER];
#pragma unroll
		for (int b = 0; b < PER; ++b) {
			const int i = tid + b * NT;
			if (i < n) v[b] = src(i);
		}
		__syncthreads();
#pragma unroll
		for (int b = 0; b < PER; ++b) {
			const int i = tid + b * NT;
			if (i < n) {
				buf[i + H] = v[b];
				if (i < H) buf[i + H + n] = v[b];
				if (i >= n - H) buf[i + H - n] = v[b];
			}
		}
		__syncthreads();
	}
	const bool even = n % 2 == 0;
	const int sp = even ? P / 2 : P;              // fine points per half with weights of their own
	const float4* w4 = p.w4 + g * sp;
	const int* q0 = p.q0 + g * sp;
	auto ld = [&](int i) -> float2 {
		const bool up = even && i >= P / 2;
		const int e = up ? i - P / 2 : i;
		const float4 w = w4[e];
		const float2* x = buf + q0[e] + (up ? n / 2 : 0) + H;
		float2 s = make_float2(w.x * x[0].x, w.x * x[0].y);
		s.x = fmaf(w.y, x[1].x, s.x); s.y = fmaf(w.y, x[1].y, s.y);
		s.x = fmaf(w.z, x[2].x, s.x); s.y = fmaf(w.z, x[2].y, s.y);
		s.x = fmaf(w.w, x[3].x, s.x); s.y = fmaf(w.w, x[3].y, s.y);
		return s;
	};
	auto st = [&](int i, float2 v) { hb[i] = v; };
	fft_lds_io<P, HT, false>(hb, p.tw, lt, ld, st);
	const int kmax = n / 2;
	float2 v[PER];
#pragma unroll
	for (int b = 0; b < PER; ++b) {
		const int i = tid + b * NT;
		if (i < n) {
			const int k = i <= kmax ? i : i - n;
			const int a = k < 0 ? -k : k, l = k & (P - 1);
			const float2 e = buf[l], o = buf[RL + l];
			const float d = p.mode[a].x;
			const float2 f = p.mode[kmax + 1 + a];
			const float2 t = k < 0 ? cmul(o, f) : cmulc(o, f);
			v[b] = make_float2(fmaf(e.x, d, t.x), fmaf(e.y, d, t.y));
		}
	}
	__syncthreads();
#pragma unroll
	for (int b = 0; b < PER; ++b) {
		const int i = tid + b * NT;
		if (i < n) buf[pidx(i)] = v[b];
	}
	__syncthreads();
}

// ---- any length ------------------------------------------------------------
// Forward transform of src(i), i in [0, n), result in logical buf[0..n).
// src may read buf.
template <int NT, int MAXN, class Src>
__device__ __forceinline__ void fft_any_fwd(float2* buf, const Fft1dPlan& p, int tid, const Src& src)
{
	if (p.mode != nullptr) {
		itp_fwd<NT, MAXN>(buf, p, tid, src);
	} else if (p.nrad == 0 && p.n == MAXN) {
		fft_lds_io<MAXN, NT, false>(buf, p.tw, tid, src, LdsOut{buf});
	} else if (p.nrad == 0 && p.n == MAXN / 2) {
		fft_lds_io<MAXN / 2, NT, false>(buf, p.tw, tid, src, LdsOut{buf});
	} else if (p.nrad > 0) {
		fft_mixed<NT, MAXN, false>(buf, p, tid, src);
	} else {
		constexpr int PER = (MAXN + NT - 1) / NT;
		float2 v[PER];
#pragma unroll
		for (int b = 0; b < PER; ++b) {
			const int i = tid + b * NT;
			if (i < p.n) v[b] = src(i);
		}
		__syncthreads();
#pragma unroll
		for (int b = 0; b < PER; ++b) {
			const int i = tid + b * NT;
			if (i < p.n) buf[pidx(i)] = v[b];
		}
		__syncthreads();
		fft_lds_rt<NT, MAXN, false>(buf, p.n, p.tw, tid);
	}
}

// Inverse transform of the modes src(k), k in (-n/2, n/2].  src may read buf.
template <int NT, int MAXN, class Src>
__device__ __forceinline__ void fft_inv_passes(float2* buf, const Fft1dPlan& p, int tid, const Src& src)
{
	if (p.nrad > 0) {
		fft_mixed<NT, MAXN, true>(buf, p, tid, [&](int i) -> float2 { return src(i > p.n / 2 ? i - p.n : i); });
		return;
	}
	constexpr int PER = (MAXN + NT - 1) / NT;
	float2 v[PER];
#pragma unroll
	for (int b = 0; b < PER; ++b) {
		const int i = tid + b * NT;
		if (i < p.n) v[b] = src(i > p.n / 2 ? i - p.n : i);
	}
	__syncthreads();
#pragma unroll
	for (int b = 0; b < PER; ++b) {
		const int i = tid + b * NT;
		if (i < p.n) buf[pidx(i)] = v[b];
	}
	__syncthreads();
	fft_lds_rt<NT, MAXN, true>(buf, p.n, p.tw, tid);
}

// Every output t handed to out(t, v) once; out may not write buf.
template <int NT, int MAXN, class Src, class Out>
__device__ __forceinline__ void fft_any_inv(float2* buf, const Fft1dPlan& p, int tid, const Src& src, const Out& out)
{
	if (p.mode != nullptr) {
		itp_inv<NT, MAXN, false>(buf, p, tid, src, out);
		return;
	}
	fft_inv_passes<NT, MAXN>(buf, p, tid, src);
	for (int i = tid; i < p.n; i += NT) out(i, buf[pidx(i)]);
}

// Result in logical buf[0..n), visible to the workgroup.
template <int NT, int MAXN, class Src>
__device__ __forceinline__ void fft_any_inv_lds(float2* buf, const Fft1dPlan& p, int tid, const Src& src)
{
	if (p.mode != nullptr) {
		itp_inv<NT, MAXN, true>(buf, p, tid, src, LdsOut{buf});
		__syncthreads();
		return;
	}
	fft_inv_passes<NT, MAXN>(buf, p, tid, src);
}

}  // namespace gctf
