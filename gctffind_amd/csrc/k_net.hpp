// k_net.hpp -- BF16 kernels of the defocus-proposal network: five launches
// for a forward pass, ten for a training step.
//
// The layers are too small to fill the chip one matrix at a time (conv2 of a
// batch of 256 is 1.9 GFLOP), so what bounds them is launches and passes over
// memory, not the matrix cores.  Every convolution is an implicit GEMM: the
// input tile goes to LDS once as BF16 and the 7 taps are 7 shifted reads of
// it; no column matrix exists.  Bias, ReLU and pooling are the epilogue, the
// backward pass of pooling and ReLU the prologue of the gradients, which need
// one bit per activation (its sign) and not the activation.  All weight
// gradients are one launch, split over the batch, and one reduction in a
// fixed order, so training stays deterministic.  Operands are rounded to BF16
// where they enter the matrix cores; sums, activations, gradients and
// parameters are FP32 throughout.
//
// Every sum is formed in the order of the plain im2col GEMM with its K splits
// (gemm_splits): an activation that differs in its last bit rounds to another
// BF16 value or changes sign now and then, and a gradient then differs by
// 1e-3, as if it had come from other inputs.
//
// A training step of 256 spectra took 1030 us of kernel time as im2col GEMMs
// (44 launches).
//
// MFMA layout (v_mfma_f32_32x32x16_bf16, wave64): lane l holds
// A[l % 32][8 (l / 32) + j] and B[8 (l / 32) + j][l % 32], j = 0..7; result
// register r of lane l is D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#pragma once
#include "gctf_net.hpp"

namespace gctf {

typedef __bf16 nbf16x8 __attribute__((ext_vector_type(8)));
typedef float nfloatx16 __attribute__((ext_vector_type(16)));
typedef unsigned int nuintx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int mfma_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

__device__ __forceinline__ unsigned int pack_bf16(float a, float b)
{
	const __bf16 x = (__bf16)a, y = (__bf16)b;
	return (unsigned int)__builtin_bit_cast(unsigned short, x)
		| ((unsigned int)__builtin_bit_cast(unsigned short, y) << 16);
}

// ---------------------------------------------------------------------------
// Weights as MFMA fragments, rounded once per pass: fragment f is 64 lanes of
// 8 BF16 values, one coalesced 16-byte load per lane.
//   conv layer l forward: (2 l * 28 + s) * 2 + mt: rows m = 32 mt + lane % 32
//     of W[m][k], k = 16 s + 8 (lane / 32) + j (= 7 channel + tap)
//   its input gradient: ((2 l + 1) * 28 + 4 t + s) * 2 + mt: rows m of
//     W[k][m][t], k = 16 s + 8 (lane / 32) + j
//   fc1 forward (A): kFragFc1 + kt * 4 + jt: W5[32 jt + lane % 32][16 kt + 8 h + j]
//   fc1 input gradient (B): kFragFc1Back + kt * 8 + js:
//     W5[16 js + 8 h + j][32 kt + lane % 32]
// ---------------------------------------------------------------------------
constexpr int kConvSlices = kNetCol / 16;                  // K slices of 16
constexpr int kFragConv = kConvSlices * 2;                 // fragments of a layer and direction
constexpr int kFragFc1 = 6 * kFragConv;
constexpr int kFragFc1Count = (kNetFlat / 16) * (kNetHidden / 32);
constexpr int kFragFc1Back = kFragFc1 + kFragFc1Count;
constexpr int kFragTotal = kFragFc1Back + kFragFc1Count;

// Fragments 4 block .. + 3, a wave each; directions 1 only when back.
__device__ __forceinline__ void net_weights(const float* __restrict__ prm, int back, uint4* __restrict__ frag, int block)
{
	const int f = block * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
	const int row = lane & 31, h = lane >> 5;
	if (f >= (back ? kFragTotal : kFragFc1Back)) return;
	float v[8];
	if (f < kFragFc1) {
		const int mt = f & 1, i = (f >> 1) % kConvSlices, d = (f / kFragConv) & 1, l = f / (2 * kFragConv);
		if (d == 1 && !back) return;
		const float* w = prm + (l == 0 ? kNetW2 : l == 1 ? kNetW3 : kNetW4);
		const int m = 32 * mt + row;
		if (d == 0) {
#pragma unroll
			for (int j = 0; j < 8; ++j) v[j] = w[(long long)m * kNetCol + 16 * i + 8 * h + j];
		} else {
			const int t = i >> 2, k = 16 * (i & 3) + 8 * h;
#pragma unroll
			for (int j = 0; j < 8; ++j) v[j] = w[(long long)(k + j) * kNetCol + m * kNetTaps + t];
		}
	} else if (f < kFragFc1Back) {
		const int i = f - kFragFc1, jt = i & 3, kt = i >> 2;
		const float* w = prm + kNetW5 + (long long)(32 * jt + row) * kNetFlat + 16 * kt + 8 * h;
#pragma unroll
		for (int j = 0; j < 8; ++j) v[j] = w[j];
	} else {
		const int i = f - kFragFc1Back, js = i & 7, kt = i >> 3;
		const float* w = prm + kNetW5 + (long long)(16 * js + 8 * h) * kNetFlat + 32 * kt + row;
#pragma unroll
		for (int j = 0; j < 8; ++j) v[j] = w[(long long)j * kNetFlat];
	}
	frag[(long long)f * 64 + lane] = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]),
		pack_bf16(v[6], v[7]));
}

__device__ __forceinline__ nbf16x8 load_frag(const uint4* __restrict__ frag, int f, int lane)
{
	return __builtin_bit_cast(nbf16x8, frag[(long long)f * 64 + lane]);
}

// ---------------------------------------------------------------------------
// Input z-score, conv1 (1 -> 64, 7 taps), bias, ReLU and pool of spectrum b;
// thread = pooled position, half of the channels.  a1 the pooled outputs, m1 the
// signs of the two pooled activations (bits 0 and 1).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void net_front(const float* __restrict__ radial, int ld,
	const float* __restrict__ prm, int B, float* __restrict__ x0, float* __restrict__ a1,
	unsigned char* __restrict__ m1, int b)
{
	__shared__ double r1[256], r2[256];
	__shared__ float xs[kNetBins + 8];
	__shared__ float ws[kNetCh * (kNetTaps + 1)];         // weights, then biases
	const int t = threadIdx.x;
	for (int i = t; i < kNetCh * (kNetTaps + 1); i += 256) ws[i] = prm[kNetW1 + i];
	static_assert(kNetB1 == kNetW1 + kNetCh * kNetTaps, "weights and biases are neighbours");
	const float v = radial[(long long)b * ld + t];
	const bool use = t >= kNetBin0;
	r1[t] = use ? (double)v : 0.0;
	r2[t] = use ? (double)v * v : 0.0;
	__syncthreads();
	for (int s = 128; s > 0; s >>= 1) {
		if (t < s) { r1[t] += r1[t + s]; r2[t] += r2[t + s]; }
		__syncthreads();
	}
	const double cnt = (double)(kNetBins - kNetBin0);
	const double mean = r1[0] / cnt;
	const double var = fmax(r2[0] / cnt - mean * mean, 1e-24);
	const float x = use ? (float)(((double)v - mean) / sqrt(var)) : 0.f;
	if (m1) x0[(long long)b * kNetBins + t] = x;
	xs[t + 3] = x;
	if (t < 3) xs[t] = 0.f;
	if (t >= kNetBins - 5) xs[t + 8] = 0.f;
	__syncthreads();
	constexpr int L2 = kNetBins / 2;
	const int p = t % L2;
	float win[kNetTaps + 1];
#pragma unroll
	for (int i = 0; i <= kNetTaps; ++i) win[i] = xs[2 * p + i];
	const int c0 = t / L2;
#pragma unroll 4
	for (int c = c0; c < kNetCh; c += 2) {
		const float* w = ws + c * kNetTaps;
		float y[2];
#pragma unroll
		for (int q = 0; q < 2; ++q) {
			float z = ws[kNetCh * kNetTaps + c];
#pragma unroll
			for (int i = 0; i < kNetTaps; ++i) z = fmaf(w[i], win[i + q], z);
			y[q] = fmaxf(z, 0.f);
		}
		const long long o = ((long long)c * B + b) * L2 + p;
		a1[o] = 0.5f * (y[0] + y[1]);
		if (m1) m1[o] = (unsigned char)((y[0] > 0.f ? 1 : 0) | (y[1] > 0.f ? 2 : 0));
	}
}

// The pass's first launch: workgroups 0 .. B - 1 a spectrum each, the others the
// weight fragments, which only the following launches read.  Launches of their own
// cost proposals of 32 spectra 4 us of 77.
__global__ __launch_bounds__(256) void k_net_front(const float* __restrict__ radial, int ld,
	const float* __restrict__ prm, int B, float* __restrict__ x0, float* __restrict__ a1,
	unsigned char* __restrict__ m1, int back, uint4* __restrict__ frag)
{
	const int b = blockIdx.x;
	if (b < B) net_front(radial, ld, prm, B, x0, a1, m1, b);
	else net_weights(prm, back, frag, b - B);
}

// ---------------------------------------------------------------------------
// A 64 -> 64 channel, 7-tap convolution over rows of length L (zero padding
// 3) as an implicit GEMM, K = 7 channel + tap: input a [64][B L], output bias +
// ReLU + pool in out [64][B L / 2], the signs in sgn (when not null).  A
// workgroup takes 128 positions, a wave 64 channels x 32 of them (an input
// fragment serves two MFMAs), or 64 positions and 32 x 32.  LDS holds a channel's positions in a
// row (each row segment with its halo of 3 on either side): the taps of a
// position are neighbours, and 8 consecutive k are at most two runs, at
// addresses that are constants but for the lane's half: k + 8 is the next
// channel's next tap, or the channel's after that first one.
// A sum of K is formed in splits of SPL slices of 16 (gemm_splits), a template
// parameter: with a runtime count each slice ended in a branch, and its weight
// fragments were loaded where they were used, 24 us for any batch.
// ---------------------------------------------------------------------------
template <int NW, int SPL, int L>
__global__ __launch_bounds__(256) void k_net_conv(const float* __restrict__ a, const uint4* __restrict__ frag,
	const float* __restrict__ bias, int BL, float* __restrict__ out, unsigned char* __restrict__ sgn)
{
	constexpr int TN = 32 * NW;
	constexpr int MW = NW == 4 ? 2 : 1;                  // 32-channel tiles per wave
	constexpr int seg = L < TN ? L : TN, pitch = seg + 6, pairs = TN / seg * (pitch / 2);
	constexpr int PT = 2 * pairs + 2;
	__shared__ __attribute__((aligned(16))) unsigned short xs[kNetCh * PT];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int row = lane & 31, h = lane >> 5;
	const int q0 = blockIdx.x * TN;
	const int m0 = NW == 4 ? 0 : wave >> 1;
	// the loads of 6 passes over the tile in flight at once
#pragma unroll 6
	for (int i = tid; i < pairs * kNetCh; i += 256) {
		const int ci = i / pairs, r = (i - ci * pairs) * 2;
		const int sg = r / pitch, o = r - sg * pitch - 3;
		const int qs = q0 + sg * seg;
		float v[2];
#pragma unroll
		for (int j = 0; j < 2; ++j) {
			const int l = qs % L + o + j;                     // place in its row
			const bool in = l >= 0 && l < L && qs < BL;
			const float x = a[(long long)ci * BL + (in ? qs + o + j : 0)];
			v[j] = in ? x : 0.f;
		}
		*reinterpret_cast<unsigned int*>(xs + ci * PT + r) = pack_bf16(v[0], v[1]);
	}
	const int p = (NW == 4 ? wave : wave & 1) * 32 + row; // position in the tile
	const int sg = p / seg;
	const unsigned short* base = xs + sg * pitch + p - sg * seg;
	const unsigned short* b1 = base + h * (PT + 1);       // k + 8 one channel and one tap on
	const unsigned short* b2 = base + h * (2 * PT - 6);   // from tap 6: two channels on, tap 0
	nfloatx16 acc[MW], tot[MW];
#pragma unroll
	for (int m = 0; m < MW; ++m)
#pragma unroll
		for (int r = 0; r < 16; ++r) { acc[m][r] = 0.f; tot[m][r] = 0.f; }
	// weight fragments of G slices ahead
	constexpr int G = 4;
	static_assert(kConvSlices % G == 0, "whole groups of slices");
	nbf16x8 wc[MW * G], wx[MW * G];
#pragma unroll
	for (int i = 0; i < MW * G; ++i) wc[i] = load_frag(frag, i / MW * 2 + m0 + i % MW, lane);
	__syncthreads();
#pragma unroll
	for (int s = 0; s < kConvSlices; ++s) {
		if (s % G == 0 && s + G < kConvSlices)
#pragma unroll
			for (int i = 0; i < MW * G; ++i) wx[i] = load_frag(frag, (s + G + i / MW) * 2 + m0 + i % MW, lane);
		unsigned int u[4];
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			const int k = 16 * s + j, t = k % kNetTaps;
			const unsigned int e = (t < kNetTaps - 1 ? b1 : b2)[(k / kNetTaps) * PT + t];
			if (j % 2 == 0) u[j / 2] = e;
			else u[j / 2] |= e << 16;
		}
		const nbf16x8 x = __builtin_bit_cast(nbf16x8, make_uint4(u[0], u[1], u[2], u[3]));
#pragma unroll
		for (int m = 0; m < MW; ++m)
			acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wc[MW * (s % G) + m], x, acc[m], 0, 0, 0);
		if (s % G == G - 1)
#pragma unroll
			for (int i = 0; i < MW * G; ++i) wc[i] = wx[i];
		if ((s + 1) % SPL == 0 || s == kConvSlices - 1) {
#pragma unroll
			for (int m = 0; m < MW; ++m)
#pragma unroll
				for (int r = 0; r < 16; ++r) { tot[m][r] += acc[m][r]; acc[m][r] = 0.f; }
		}
	}
	const int q = q0 + p;
#pragma unroll
	for (int m = 0; m < MW; ++m)
#pragma unroll
		for (int r = 0; r < 16; ++r) {
			const int c = 32 * (m0 + m) + mfma_row(r, h);
			const float y = fmaxf(tot[m][r] + bias[c], 0.f);
			const float y1 = __shfl_xor(y, 1);
			if ((lane & 1) == 0 && q < BL) {
				const long long o = (long long)c * (BL / 2) + (q >> 1);
				out[o] = 0.5f * (y + y1);
				if (sgn) sgn[o] = (unsigned char)((y > 0.f ? 1 : 0) | (y1 > 0.f ? 2 : 0));
			}
		}
}

// The input gradient of the layer: dA[ci][q] = sum over taps t (in that order,
// FP32) of sum over co of W[co][ci][t] dZ[co][q - t + 3], with dZ = (sign)
// 0.5 dP of the layer's pooled gradient dP [64][B L / 2] and signs sin.  64
// channels x 64 NS positions per workgroup, each wave 32 x 32 NS.  LDS row =
// position (each segment with its halo), 64 channels of BF16 and 16 bytes of
// padding: a tap's fragment is the same rows shifted by the tap, 16-byte reads
// that spread over all banks.
constexpr int kConvPitch = kNetCh + 8;

template <int NS, int L>
__global__ __launch_bounds__(256) void k_net_conv_back(const float* __restrict__ dP,
	const unsigned char* __restrict__ sin, const uint4* __restrict__ frag, int BL, float* __restrict__ out)
{
	constexpr int TN = 64 * NS;
	constexpr int seg = L < TN ? L : TN, pitch = seg + 6, rows = TN / seg * pitch;
	__shared__ __attribute__((aligned(16))) __bf16 xs[rows * kConvPitch];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int row = lane & 31, h = lane >> 5;
	const int mt = wave >> 1, wn = wave & 1;
	const int q0 = blockIdx.x * TN;
#pragma unroll 2
	for (int i = tid; i < rows * (kNetCh / 8); i += 256) {
		const int cg = i / rows, r = i - cg * rows;
		const int sg = r / pitch, o = r - sg * pitch - 3;
		const int qs = q0 + sg * seg, q = qs + o;
		const int l = qs % L + o;                            // place in its row
		const bool in = l >= 0 && l < L && qs < BL;
		const long long H = BL / 2;
		const long long e = in ? q >> 1 : 0;
		float v[8];
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			const long long k = (cg * 8 + j) * H + e;
			const int on = (sin[k] >> (q & 1)) & 1;
			const float d = 0.5f * dP[k];
			v[j] = in && on ? d : 0.f;
		}
		*reinterpret_cast<uint4*>(xs + r * kConvPitch + cg * 8) = make_uint4(pack_bf16(v[0], v[1]),
			pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
	}
	__syncthreads();
	nfloatx16 tot[NS];
	int base[NS];
#pragma unroll
	for (int n = 0; n < NS; ++n) {
#pragma unroll
		for (int r = 0; r < 16; ++r) tot[n][r] = 0.f;
		const int p = (wn * NS + n) * 32 + row;           // position in the tile
		const int sg = p / seg;
		base[n] = (sg * pitch + p - sg * seg) * kConvPitch + 8 * h;
	}
#pragma unroll
	for (int t = 0; t < kNetTaps; ++t) {
		nfloatx16 acc[NS];
#pragma unroll
		for (int n = 0; n < NS; ++n)
#pragma unroll
			for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
#pragma unroll
		for (int s = 0; s < 4; ++s) {
			const nbf16x8 w = load_frag(frag, (t * 4 + s) * 2 + mt, lane);
#pragma unroll
			for (int n = 0; n < NS; ++n) {
				const nbf16x8 x = *reinterpret_cast<const nbf16x8*>(xs + base[n] + (kNetTaps - 1 - t) * kConvPitch + 16 * s);
				acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, acc[n], 0, 0, 0);
			}
		}
#pragma unroll
		for (int n = 0; n < NS; ++n)
#pragma unroll
			for (int r = 0; r < 16; ++r) tot[n][r] += acc[n][r];
	}
#pragma unroll
	for (int n = 0; n < NS; ++n) {
		const int q = q0 + (wn * NS + n) * 32 + row;
		if (q < BL)
#pragma unroll
			for (int r = 0; r < 16; ++r) out[(long long)(32 * mt + mfma_row(r, h)) * BL + q] = tot[n][r];
	}
}

// ---------------------------------------------------------------------------
// fc1, ReLU, fc2 of 32 spectra per workgroup (16 waves: 4 hidden tiles x 4
// quarters of the 1024 inputs), and with target the loss, its gradient and the
// gradients of the hidden layer (dh [128][B]) and of the pooled conv4 output
// (dA4 [64][B 16]).
// Loss per spectrum and its gradient (divided by B).  target[b] =
// (mean defocus A, astigmatism A, azimuth deg, confidence label).
//   100 (o0 - ln(df / 1e4))^2 + 0.25 (o1 - ast / 1e3)^2
//   + 0.05 (1 - cos 2 (o2 - az)) + 0.5 w BCE(sigmoid(o3), c)
// The label is measured on the micrograph (whether the learned path's
// narrowed search ended within 20 A of the full search): > 0 gives c = 1,
// < 0 gives c = 0, and 0 (unlabelled) drops the confidence term (w = 0).
// spl1, spl2: K slices per split of the two products' sums (gemm_splits).
// ---------------------------------------------------------------------------
__device__ __forceinline__ float net_loss(const float* ob, const float* tb, int B, float* dO)
{
	const float y0 = logf(tb[0] * 1.0e-4f), y1 = tb[1] * 1.0e-3f;
	const float az = tb[2] * 0.017453292519943295f;
	const float e0 = ob[0] - y0, e1 = ob[1] - y1;
	const float d2 = 2.0f * (ob[2] - az);
	const float c = tb[3] > 0.0f ? 1.0f : 0.0f;
	const float w = tb[3] != 0.0f ? 1.0f : 0.0f;
	const float x = ob[3];
	// softplus forms of the log-sigmoid terms
	const float sp_pos = fmaxf(x, 0.f) + log1pf(expf(-fabsf(x)));   // -log(1 - p)
	const float sp_neg = sp_pos - x;                                 // -log p
	const float bce = c * sp_neg + (1.0f - c) * sp_pos;
	const float p = 1.0f / (1.0f + expf(-x));
	const float inv = 1.0f / (float)B;
	dO[0] = 200.0f * e0 * inv;
	dO[1] = 0.5f * e1 * inv;
	dO[2] = 0.1f * sinf(d2) * inv;
	dO[3] = 0.5f * w * (p - c) * inv;
	return 100.0f * e0 * e0 + 0.25f * e1 * e1 + 0.05f * (1.0f - cosf(d2)) + 0.5f * w * bce;
}

__global__ __launch_bounds__(1024) void k_net_fc(const float* __restrict__ a4, const uint4* __restrict__ frag,
	const float* __restrict__ prm, int B, int spl1, int spl2, float* __restrict__ o, const float* __restrict__ target,
	float* __restrict__ h, float* __restrict__ dO, double* __restrict__ lpart, float* __restrict__ dh,
	float* __restrict__ dA4)
{
	constexpr int NB = 32, LD = NB + 1, HP = kNetHidden + 8;
	__shared__ float hs[kNetHidden * LD];
	__shared__ float os[NB][kNetOut], ds[NB][kNetOut];
	__shared__ float w6[kNetOut * (kNetHidden + 1)];        // fc2's weights, then its biases
	static_assert(kNetB6 == kNetW6 + kNetOut * kNetHidden, "weights and biases are neighbours");
	__shared__ __attribute__((aligned(16))) __bf16 dhs[NB * HP];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int row = lane & 31, hf = lane >> 5;
	const int b0 = blockIdx.x * NB;
	// the tile's inputs, read once for the four hidden tiles: row = spectrum
	constexpr int XP = kNetFlat + 8;
	__shared__ __attribute__((aligned(16))) __bf16 fs[NB * XP];
#pragma unroll
	for (int i = 0; i < kNetFlat * NB / 4 / 1024; ++i) {
		const int e = tid + i * 1024, q = e % 4, b = e / 4 % NB, c = e / (4 * NB);
		const float4 v = *reinterpret_cast<const float4*>(a4 + ((long long)c * B + min(b0 + b, B - 1)) * kNetL4 + 4 * q);
		*reinterpret_cast<uint2*>(fs + b * XP + c * kNetL4 + 4 * q) = make_uint2(pack_bf16(v.x, v.y), pack_bf16(v.z, v.w));
	}
	if (tid < kNetOut * (kNetHidden + 1)) w6[tid] = prm[kNetW6 + tid];
	{
		// quarter ks of the slices to wave group ks, where it holds whole splits
		// (of 4, 8 or 16 slices: batches up to 1024, of 1601 to 2048 and of 3265
		// to 4096); else group 0 takes them all.  A forward pass of 1030 spectra
		// (splits of 5) takes 149 us, of 1700 (splits of 8) 154 us
		const int jt = wave & 3, ks = wave >> 2;
		constexpr int NK = kNetFlat / 16, QK = NK / 4;
		auto slice = [&](int c, nfloatx16 acc) {             // channel c: inputs 16 c .. 16 c + 15
			const nbf16x8 x = *reinterpret_cast<const nbf16x8*>(fs + row * XP + c * kNetL4 + 8 * hf);
			return __builtin_amdgcn_mfma_f32_32x32x16_bf16(load_frag(frag, kFragFc1 + c * 4 + jt, lane), x, acc, 0, 0, 0);
		};
		__syncthreads();
		nfloatx16 zero, acc;
#pragma unroll
		for (int r = 0; r < 16; ++r) zero[r] = 0.f;
		auto at = [&](int r) -> float& { return hs[(jt * 32 + mfma_row(r, hf)) * LD + row]; };
		if (spl1 >= 4 && QK % spl1 == 0) {
			nfloatx16 part[4];                                // splits of 4 slices; wider ones end in every second or fourth
			acc = zero;
#pragma unroll
			for (int i = 0; i < QK; ++i) {
				acc = slice(ks * QK + i, acc);
				if (i % 4 == 3) {
					part[i / 4] = acc;
					if ((i + 1) % spl1 == 0) acc = zero;
				}
			}
			for (int g = 0; g < 4; ++g) {
				if (ks == g) {
#pragma unroll
					for (int i = 0; i < 4; ++i)
						if ((4 * i + 4) % spl1 == 0) {
							const bool first = g == 0 && 4 * i + 4 == spl1;
#pragma unroll
							for (int r = 0; r < 16; ++r) at(r) = first ? part[i][r] : at(r) + part[i][r];
						}
				}
				__syncthreads();
			}
		} else {
			if (ks == 0) {
				nfloatx16 tot = zero;
				acc = zero;
				for (int c = 0; c < NK; ++c) {
					acc = slice(c, acc);
					if ((c + 1) % spl1 == 0 || c == NK - 1) { tot += acc; acc = zero; }
				}
#pragma unroll
				for (int r = 0; r < 16; ++r) at(r) = tot[r];
			}
			__syncthreads();
		}
	}
	for (int i = tid; i < kNetHidden * NB; i += 1024) {
		const int j = i / NB, b = i % NB, k = j * LD + b;
		const float v = fmaxf(hs[k] + prm[kNetB5 + j], 0.f);
		hs[k] = v;
		if (target && b0 + b < B) h[(long long)j * B + b0 + b] = v;
	}
	__syncthreads();
	if (tid < NB * kNetOut) {
		const int k = tid / NB, b = tid % NB;
		const float* w = w6 + k * kNetHidden;
		float s = w6[kNetOut * kNetHidden + k];
#pragma unroll 16
		for (int j = 0; j < kNetHidden; ++j) s = fmaf(w[j], hs[j * LD + b], s);
		os[b][k] = s;
		if (b0 + b < B) o[(long long)(b0 + b) * kNetOut + k] = s;
	}
	if (!target) return;
	__syncthreads();
	if (tid < NB) {
		const int b = b0 + tid;
		const float l = net_loss(os[tid], target + (long long)min(b, B - 1) * 4, B, ds[tid]);
		if (b < B) {
			lpart[b] = (double)l;
#pragma unroll
			for (int k = 0; k < kNetOut; ++k) dO[(long long)b * kNetOut + k] = ds[tid][k];
		}
	}
	__syncthreads();
	for (int i = tid; i < kNetHidden * NB; i += 1024) {
		const int j = i / NB, b = i % NB;
		float s = 0.f;
#pragma unroll
		for (int k = 0; k < kNetOut; ++k) s = fmaf(w6[k * kNetHidden + j], ds[b][k], s);
		s = hs[j * LD + b] > 0.f ? s : 0.f;
		if (b0 + b < B) dh[(long long)j * B + b0 + b] = s;
		dhs[b * HP + j] = (__bf16)s;
	}
	__syncthreads();
	// dF[b][k] = sum_j dh[b][j] W5[j][k], k = 16 c + l
#pragma unroll
	for (int q = 0; q < 2; ++q) {
		const int kt = wave * 2 + q;
		nfloatx16 acc, tot;
#pragma unroll
		for (int r = 0; r < 16; ++r) { acc[r] = 0.f; tot[r] = 0.f; }
#pragma unroll
		for (int js = 0; js < 8; ++js) {
			acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
				*reinterpret_cast<const nbf16x8*>(dhs + row * HP + 16 * js + 8 * hf),
				load_frag(frag, kFragFc1Back + kt * 8 + js, lane), acc, 0, 0, 0);
			if ((js + 1) % spl2 == 0 || js == 7)
#pragma unroll
				for (int r = 0; r < 16; ++r) { tot[r] += acc[r]; acc[r] = 0.f; }
		}
		const int k = kt * 32 + row, c = k / kNetL4, l = k % kNetL4;
#pragma unroll
		for (int r = 0; r < 16; ++r) {
			const int b = b0 + mfma_row(r, hf);
			if (b < B) dA4[((long long)c * B + b) * kNetL4 + l] = tot[r];
		}
	}
}

// ---------------------------------------------------------------------------
// All parameter gradients: one launch over the work of every layer (they only
// read what the passes before left), one workgroup per item.
// ---------------------------------------------------------------------------
constexpr int kDwChunk = 128;       // positions per LDS tile

struct NetDwArgs {
	int B;
	// conv2..4: layer input a [64][B L], pooled gradient dA [64][B L / 2],
	// signs; positions per split and splits of the weight gradient's sum
	const float* a[3];
	const float* dA[3];
	const unsigned char* sgn[3];
	int ksplit[3], splits[3];
	float* part[3];                   // [split][64][448]
	// conv1
	const float *x0, *dA1;
	const unsigned char* m1;
	// fc1, fc2; batch per split of fc1's weight gradient
	const float *a4, *dh, *h, *dO;
	int ksplit5;
	const double* lpart;
	float* grad;
	double* loss;
	// first item of each kind: conv2..4, conv1, conv2..4 biases, fc1, fc2
	int first[7];
};

__device__ __forceinline__ float net_dz(float d, int sign) { return sign ? 0.5f * d : 0.f; }

// Gradient of a conv layer's weights over one split of the positions:
// dW[co][ci][t] = sum_q dZ[co][q] a[ci][q + t - 3].  K = positions, in slices
// of 16, each within one row; wave (co half, ci half) keeps the 32 x 32 tiles
// of the 7 taps.  In LDS both operands have positions along the row; a slice
// of a is 24 values from 3 positions early on, so that the 16 around a lane's
// 8 positions are two aligned 16-byte reads and the taps are their 7 shifts.
constexpr int kDwZ = kDwChunk + 8, kDwA = kDwChunk / 16 * 24 + 8;   // odd multiples of 8: all banks
template <int layer>
__device__ __forceinline__ void net_dw_conv(const NetDwArgs& g, int split, __bf16* sm)
{
	constexpr int L = kNetBins / 2 >> layer;
	const int BL = g.B * L;
	const float* a = g.a[layer];
	const float* dA = g.dA[layer];
	const unsigned char* sg = g.sgn[layer];
	__bf16* zs = sm;
	__bf16* as = sm + kNetCh * kDwZ;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int row = lane & 31, h = lane >> 5;
	const int wm = wave >> 1, wn = wave & 1;
	nfloatx16 acc[kNetTaps];
#pragma unroll
	for (int t = 0; t < kNetTaps; ++t)
#pragma unroll
		for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
	const int qe = min(BL, (split + 1) * g.ksplit[layer]);       // BL, ksplit: multiples of 16
	for (int q0 = split * g.ksplit[layer]; q0 < qe; q0 += kDwChunk) {
		// dZ: 64 channels x 16 groups of 8 positions, 4 per thread
#pragma unroll
		for (int i = 0; i < 4; ++i) {
			const int co = (tid >> 4) + 16 * i, pg = tid & 15;
			const int q = q0 + 8 * pg;
			const bool in = q < qe;
			float v[8];
			const long long e = (long long)co * (BL / 2) + (in ? q >> 1 : 0);
#pragma unroll
			for (int p = 0; p < 4; ++p) {
				const int s = in ? sg[e + p] : 0;
				const float d = dA[e + p];
				v[2 * p] = net_dz(d, s & 1);
				v[2 * p + 1] = net_dz(d, s & 2);
			}
			*reinterpret_cast<uint4*>(zs + co * kDwZ + 8 * pg) = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]),
				pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
		}
		// a: 64 channels x 8 slices x 3 groups of 8, 6 per thread
#pragma unroll
		for (int n = 0; n < kNetCh * 24 / 256; ++n) {
			const int i = tid + n * 256;
			const int ci = i / 24, gr = i - ci * 24, s = gr / 3;
			const int qs = q0 + 16 * s, o = (gr - 3 * s) * 8 - 3;
			const int l0 = qs % L + o;                           // place in its row
			float v[8];
#pragma unroll
			for (int j = 0; j < 8; ++j) {
				const bool in = l0 + j >= 0 && l0 + j < L && qs < qe;
				const float x = a[(long long)ci * BL + (in ? qs + o + j : 0)];
				v[j] = in ? x : 0.f;
			}
			*reinterpret_cast<uint4*>(as + ci * kDwA + 8 * gr) = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]),
				pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
		}
		__syncthreads();
		const int slices = min(kDwChunk, qe - q0) / 16;
		for (int s = 0; s < slices; ++s) {
			const nbf16x8 z = *reinterpret_cast<const nbf16x8*>(zs + (wm * 32 + row) * kDwZ + 16 * s + 8 * h);
			const nuintx4* w = reinterpret_cast<const nuintx4*>(as + (wn * 32 + row) * kDwA + 24 * s + 8 * h);
			const nuintx4 lo = w[0], hi = w[1];
			const unsigned int d[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
			for (int t = 0; t < kNetTaps; ++t) {
				nuintx4 u;
#pragma unroll
				for (int j = 0; j < 4; ++j)
					u[j] = t & 1 ? __builtin_amdgcn_alignbit(d[t / 2 + j + 1], d[t / 2 + j], 16) : d[t / 2 + j];
				acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(z, __builtin_bit_cast(nbf16x8, u), acc[t], 0, 0, 0);
			}
		}
		__syncthreads();
	}
	float* out = g.part[layer] + (long long)split * kNetCh * kNetCol;
	const int ci = wn * 32 + row;
#pragma unroll
	for (int r = 0; r < 16; ++r) {
		float* o = out + (wm * 32 + mfma_row(r, h)) * kNetCol + ci * kNetTaps;
#pragma unroll
		for (int t = 0; t < kNetTaps; ++t) o[t] = acc[t][r];
	}
}

// Sum of the 256 threads' values: t + 128, then 64, ...
template <typename T>
__device__ __forceinline__ T wg_tree(T v, T* red)
{
	const int tid = threadIdx.x;
	__syncthreads();
	red[tid] = v;
	__syncthreads();
	for (int o = 128; o > 0; o >>= 1) {
		if (tid < o) red[tid] += red[tid + o];
		__syncthreads();
	}
	return red[0];
}

// conv1, channel c: thread = position, the batch in order, the positions' sums
// in a tree.  The rows of kRows spectra are staged in LDS while the next
// ones' loads are in flight.
__device__ __forceinline__ void net_dw_conv1(const NetDwArgs& g, int c, float* sm)
{
	constexpr int kRows = 16, XP = kNetBins + 6;
	const int l = threadIdx.x, B = g.B;
	float* xs = sm;                                       // [kRows][XP]
	float s[kNetTaps + 1];
#pragma unroll
	for (int t = 0; t <= kNetTaps; ++t) s[t] = 0.f;
	float x[kRows], d[kRows];
	auto load = [&](int b0) {
#pragma unroll
		for (int i = 0; i < kRows; ++i) {
			const int b = min(b0 + i, B - 1);
			const long long k = ((long long)c * B + b) * (kNetBins / 2) + (l >> 1);
			x[i] = g.x0[(long long)b * kNetBins + l];
			d[i] = net_dz(g.dA1[k], (g.m1[k] >> (l & 1)) & 1);
		}
	};
	load(0);
	if (l < 6)
#pragma unroll
		for (int i = 0; i < kRows; ++i) xs[i * XP + (l < 3 ? l : kNetBins + l)] = 0.f;
	for (int b0 = 0; b0 < B; b0 += kRows) {
		__syncthreads();
		float dz[kRows];
#pragma unroll
		for (int i = 0; i < kRows; ++i) {
			xs[i * XP + l + 3] = x[i];
			dz[i] = b0 + i < B ? d[i] : 0.f;
		}
		__syncthreads();
		if (b0 + kRows < B) load(b0 + kRows);
#pragma unroll
		for (int i = 0; i < kRows; ++i) {
#pragma unroll
			for (int t = 0; t < kNetTaps; ++t) s[t] = fmaf(dz[i], xs[i * XP + l + t], s[t]);
			s[kNetTaps] += dz[i];
		}
	}
#pragma unroll
	for (int t = 0; t <= kNetTaps; ++t) {
		const float v = wg_tree(s[t], sm);
		if (l == 0) g.grad[t < kNetTaps ? kNetW1 + c * kNetTaps + t : kNetB1 + c] = v;
	}
}

// Bias of conv layer `layer`, channel c: thread sums positions tid, tid + 256, ...
__device__ __forceinline__ void net_db_conv(const NetDwArgs& g, int layer, int c, float* sm)
{
	const int BL = g.B * (kNetBins / 2 >> layer);
	const float* dA = g.dA[layer] + (long long)c * (BL / 2);
	const unsigned char* sg = g.sgn[layer] + (long long)c * (BL / 2);
	float s = 0.f;
#pragma unroll 8
	for (int i = threadIdx.x; i < BL; i += 256) s += net_dz(dA[i >> 1], (sg[i >> 1] >> (i & 1)) & 1);
	const float v = wg_tree(s, sm);
	if (threadIdx.x == 0) g.grad[(layer == 0 ? kNetB2 : layer == 1 ? kNetB3 : kNetB4) + c] = v;
}

// fc1: dW5[j][k] = sum_b dh[j][b] f[k][b], one 32 x 32 tile, four splits of
// the batch at a time.  f[16 c + l][b] = a4[c][b][l].
__device__ __forceinline__ void net_dw_fc1(const NetDwArgs& g, int item, float* sm)
{
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int row = lane & 31, h = lane >> 5;
	const int jt = item & 3, kt = item >> 2, B = g.B;
	const float* dh = g.dh + (long long)(jt * 32 + row) * B;
	const int k = kt * 32 + row, c = k / kNetL4, l = k % kNetL4;
	const float* f = g.a4 + (long long)c * B * kNetL4 + l;
	float tot[4] = {0.f, 0.f, 0.f, 0.f};
	for (int k0 = 0; k0 < B; k0 += 4 * g.ksplit5) {
		const int kb = k0 + wave * g.ksplit5, ke = min(B, kb + g.ksplit5);
		nfloatx16 acc;
#pragma unroll
		for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll 2
		for (int b0 = kb; b0 < ke; b0 += 16) {
			const int b = b0 + 8 * h;
			float u[8], v[8];
#pragma unroll
			for (int j = 0; j < 8; ++j) {
				const bool in = b + j < ke;
				const int bb = in ? b + j : 0;
				const float x = dh[bb], y = f[(long long)bb * kNetL4];
				u[j] = in ? x : 0.f;
				v[j] = in ? y : 0.f;
			}
			const uint4 p = make_uint4(pack_bf16(u[0], u[1]), pack_bf16(u[2], u[3]), pack_bf16(u[4], u[5]),
				pack_bf16(u[6], u[7]));
			const uint4 q = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]),
				pack_bf16(v[6], v[7]));
			acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(nbf16x8, p),
				__builtin_bit_cast(nbf16x8, q), acc, 0, 0, 0);
		}
#pragma unroll
		for (int r = 0; r < 16; ++r) sm[(wave * 16 + r) * 64 + lane] = acc[r];
		__syncthreads();
#pragma unroll
		for (int i = 0; i < 4; ++i)
			for (int z = 0; z < 4; ++z)
				if (k0 + z * g.ksplit5 < B) tot[i] += sm[z * 1024 + i * 256 + tid];
		__syncthreads();
	}
#pragma unroll
	for (int i = 0; i < 4; ++i) {
		const int r = (i * 256 + tid) >> 6;
		g.grad[kNetW5 + (long long)(jt * 32 + mfma_row(r, lane >> 5)) * kNetFlat + kt * 32 + (lane & 31)] = tot[i];
	}
}

// fc2 weights and bias: thread = (output, hidden unit) or output bias, the
// batch in order through LDS; fc1 bias: one hidden unit at a time.  Hidden
// units 8 item .. + 7; item 0 also the loss and the output biases.
__device__ __forceinline__ void net_dw_fc2(const NetDwArgs& g, int item, unsigned char* sm)
{
	constexpr int NJ = 8, NB = 256, LD = NB + 1;
	const int tid = threadIdx.x, B = g.B;
	float* hs = reinterpret_cast<float*>(sm);                // [NJ][LD]
	float* ds = hs + NJ * LD;                                // [kNetOut][LD]
	const int k = tid & 3, j = tid >> 2;                     // j < NJ: weights, j == NJ: output bias
	float s = 0.f;
	for (int b0 = 0; b0 < B; b0 += NB) {
		const int n = min(NB, B - b0);
		__syncthreads();
		if (tid < n) {
#pragma unroll
			for (int q = 0; q < NJ; ++q) hs[q * LD + tid] = g.h[(long long)(item * NJ + q) * B + b0 + tid];
#pragma unroll
			for (int q = 0; q < kNetOut; ++q) ds[q * LD + tid] = g.dO[(long long)(b0 + tid) * kNetOut + q];
		}
		__syncthreads();
		if (j < NJ) {
#pragma unroll 8
			for (int b = 0; b < n; ++b) s = fmaf(ds[k * LD + b], hs[j * LD + b], s);
		} else if (j == NJ && item == 0) {
#pragma unroll 8
			for (int b = 0; b < n; ++b) s += ds[k * LD + b];
		}
	}
	if (j < NJ) g.grad[kNetW6 + k * kNetHidden + item * NJ + j] = s;
	else if (j == NJ && item == 0) g.grad[kNetB6 + k] = s;
	for (int q = 0; q < NJ; ++q) {
		const int u = item * NJ + q;
		float v = 0.f;
		for (int b = tid; b < B; b += 256) v += g.dh[(long long)u * B + b];
		v = wg_tree(v, hs);
		if (tid == 0) g.grad[kNetB5 + u] = v;
	}
	if (item != 0) return;
	double l = 0.0;
	for (int b = tid; b < B; b += 256) l += g.lpart[b];
	l = wg_tree(l, reinterpret_cast<double*>(sm));
	if (tid == 0) g.loss[0] = l / (double)B;
}

constexpr int kDwLds = kNetCh * (kDwZ + kDwA) * 2;   // bytes, the conv layers' tiles

__global__ __launch_bounds__(256) void k_net_dw(NetDwArgs g)
{
	__shared__ __attribute__((aligned(16))) unsigned char sm[kDwLds];
	float* fs = reinterpret_cast<float*>(sm);
	const int i = blockIdx.x;
	if (i < g.first[1]) net_dw_conv<0>(g, i, reinterpret_cast<__bf16*>(sm));
	else if (i < g.first[2]) net_dw_conv<1>(g, i - g.first[1], reinterpret_cast<__bf16*>(sm));
	else if (i < g.first[3]) net_dw_conv<2>(g, i - g.first[2], reinterpret_cast<__bf16*>(sm));
	else if (i < g.first[4]) net_dw_conv1(g, i - g.first[3], fs);
	else if (i < g.first[5]) net_db_conv(g, (i - g.first[4]) / kNetCh, (i - g.first[4]) % kNetCh, fs);
	else if (i < g.first[6]) net_dw_fc1(g, i - g.first[5], fs);
	else net_dw_fc2(g, i - g.first[6], sm);
}

// The split partials of conv2..4's weights into the gradient, in split order.
__global__ __launch_bounds__(256) void k_net_dw_reduce(NetDwArgs g)
{
	constexpr int NW = kNetCh * kNetCol;
	const int i = blockIdx.x * 256 + threadIdx.x;
	if (i >= 3 * NW) return;
	const int l = i / NW, e = i - l * NW;
	const float* p = g.part[l] + e;
	float s = 0.f;
#pragma unroll 24
	for (int z = 0; z < g.splits[l]; ++z) s += p[(long long)z * NW];
	g.grad[(l == 0 ? kNetW2 : l == 1 ? kNetW3 : kNetW4) + e] = s;
}

}  // namespace gctf
