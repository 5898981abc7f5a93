// Learned cost model: a small multilayer perceptron
// (n_in -> hidden -> hidden -> n_out, ReLU, FP32) trained and evaluated on
// the GPU with this library's own kernels.  The scheduler uses it to predict
// the hit volume and run time of (partition, query batch) work units; its
// predictions only size buffers and order work, never prune any.
//
// Parameters are one flat FP32 array:
//   W1[n_in][H], b1[H], W2[H][H], b2[H], W3[H][n_out], b3[n_out]
// Loss: mean squared error over all outputs of a batch of rows.
// Optimiser: Adam (beta1 0.9, beta2 0.999, eps 1e-8).
#include "cost_model.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

using namespace tmx;

struct tm_mlp {
	uint32_t n_in = 0, h = 0, n_out = 0;
	uint64_t n_params = 0;
	float * d_p = nullptr;    // parameters
	float * d_g = nullptr;    // gradients
	float * d_m = nullptr;    // Adam first moment
	float * d_v = nullptr;    // Adam second moment
	uint64_t step = 0;
	// activations of the last batch
	uint32_t cap = 0;
	float * d_x = nullptr, * d_t = nullptr, * d_h1 = nullptr, * d_h2 = nullptr, * d_y = nullptr;
	float * d_dy = nullptr, * d_dh1 = nullptr, * d_dh2 = nullptr, * d_loss = nullptr;
	float * d_part = nullptr;   // gradient vectors of the row chunks
	uint64_t part_cap = 0;
	hipStream_t s = nullptr;

	size_t o_w1() const { return 0; }
	size_t o_b1() const { return (size_t)n_in * h; }
	size_t o_w2() const { return o_b1() + h; }
	size_t o_b2() const { return o_w2() + (size_t)h * h; }
	size_t o_w3() const { return o_b2() + h; }
	size_t o_b3() const { return o_w3() + (size_t)h * n_out; }

	void free_batch() {
		dfree(d_x); dfree(d_t); dfree(d_h1); dfree(d_h2); dfree(d_y);
		dfree(d_dy); dfree(d_dh1); dfree(d_dh2);
		cap = 0;
	}
	void release() {
		free_batch();
		dfree(d_p); dfree(d_g); dfree(d_m); dfree(d_v); dfree(d_loss); dfree(d_part);
		part_cap = 0;
		if (s) (void)hipStreamDestroy(s);
		s = nullptr;
	}
};

namespace {

// Y[n][m] = X[n][K] B[K][m], a 64 x 64 tile per workgroup and 4 x 4 per
// thread, operands in local memory 64 of K at a time, their loads all in flight
// together (16 at a time, loaded during the 16 before: a call of one row, all
// latency, 121 us; 112 so); each output adds its products in ascending order
// of K.
//   BACK false: B = W[K][m]; sums start at bias[c]; ReLU if relu
//   BACK true:  B = W[m][K] transposed; outputs whose H is not positive are 0
// Bound by its operands' bytes at the cost model's sizes: the 65536 x 64 x 64
// backward product takes 17 us, one thread per output with W's rows read a
// line per lane 283 us.
template <bool BACK>
__global__ void __launch_bounds__(256)
k_layer(const float * __restrict__ X, const float * __restrict__ W, const float * __restrict__ bias,
		const float * __restrict__ H, float * __restrict__ Y, uint32_t n, uint32_t K, uint32_t m, int relu) {
	__shared__ float s_x[64][68], s_w[64][68];
	const uint32_t tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
	const uint32_t r0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
	float acc[4][4];
#pragma unroll
	for (int j = 0; j < 4; ++j) {
		const uint32_t c = c0 + tx * 4 + j;
		const float b = !BACK && c < m ? bias[c] : 0.f;
#pragma unroll
		for (int i = 0; i < 4; ++i) acc[i][j] = b;
	}
	for (uint32_t k0 = 0; k0 < K; k0 += 64) {
		float lx[4][4], lw[4][4];
#pragma unroll
		for (uint32_t g = 0; g < 4; ++g) {   // 16 of K each
			if (k0 + g * 16 >= K) continue;
#pragma unroll
			for (uint32_t e = 0; e < 4; ++e) {
				const uint32_t x = tid + e * 256, k = k0 + g * 16 + (x & 15), r = x >> 4;   // 16 of K per row
				lx[g][e] = r0 + r < n && k < K ? X[(size_t)(r0 + r) * K + k] : 0.f;
				if (BACK) {
					lw[g][e] = c0 + r < m && k < K ? W[(size_t)(c0 + r) * K + k] : 0.f;
				} else {
					const uint32_t c = x & 63, kk = k0 + g * 16 + (x >> 6);
					lw[g][e] = c0 + c < m && kk < K ? W[(size_t)kk * m + c0 + c] : 0.f;
				}
			}
		}
		if (k0) __syncthreads();
#pragma unroll
		for (uint32_t g = 0; g < 4; ++g) {
			if (k0 + g * 16 >= K) continue;
#pragma unroll
			for (uint32_t e = 0; e < 4; ++e) {
				const uint32_t x = tid + e * 256;
				s_x[g * 16 + (x & 15)][x >> 4] = lx[g][e];
				if (BACK) s_w[g * 16 + (x & 15)][x >> 4] = lw[g][e];
				else s_w[g * 16 + (x >> 6)][x & 63] = lw[g][e];
			}
		}
		__syncthreads();
		const uint32_t kn = min(64u, K - k0);
		auto step = [&](uint32_t k) {
			const float4 x = *reinterpret_cast<const float4 *>(&s_x[k][ty * 4]);
			const float4 w = *reinterpret_cast<const float4 *>(&s_w[k][tx * 4]);
			const float xs[4] = {x.x, x.y, x.z, x.w}, ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
			for (int i = 0; i < 4; ++i)
#pragma unroll
				for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(xs[i], ws[j], acc[i][j]);
		};
		uint32_t k = 0;
		for (; k + 16 <= kn; k += 16) {
#pragma unroll
			for (uint32_t i = 0; i < 16; ++i) step(k + i);
		}
		for (; k < kn; ++k) step(k);
	}
#pragma unroll
	for (int i = 0; i < 4; ++i) {
		const uint32_t r = r0 + ty * 4 + i;
		if (r >= n) break;
#pragma unroll
		for (int j = 0; j < 4; ++j) {
			const uint32_t c = c0 + tx * 4 + j;
			if (c >= m) break;
			const size_t at = (size_t)r * m + c;
			float v = acc[i][j];
			if (BACK) v = H[at] <= 0.f ? 0.f : v;
			else if (relu && v < 0.f) v = 0.f;
			Y[at] = v;
		}
	}
}

// dY = 2 (Y - T) / (n m); loss += sum (Y - T)^2 / (n m), or = by one workgroup
// (a launch less to clear it: calls of a few rows, all launches, 5 % faster)
__global__ void __launch_bounds__(256)
k_mse(const float * __restrict__ Y, const float * __restrict__ T, float * __restrict__ dY, uint64_t cnt,
	  float * __restrict__ loss) {
	__shared__ float s[256];
	const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
	float e = 0.f;
	if (i < cnt) {
		const float d = Y[i] - T[i];
		dY[i] = 2.f * d / (float)cnt;
		e = d * d / (float)cnt;
	}
	s[threadIdx.x] = e;
	__syncthreads();
	for (int o = 128; o > 0; o >>= 1) {
		if ((int)threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
		__syncthreads();
	}
	if (threadIdx.x) return;
	if (gridDim.x == 1) *loss = s[0];
	else atomicAdd(loss, s[0]);
}

// dW[a][b] = A^T dY, db[b] = sum_rows dY over the rows of one chunk (rows
// blockIdx.z * per ...), into that chunk's gradient vector `part` + chunk *
// stride: a 64 x 64 tile of dW per workgroup, 4 x 4 per thread, 16 rows of
// the operands in local memory at a time; the first tile of k sums db.
// k_sum_chunks adds the chunks: one thread's walk over all 65536 rows left
// most of the chip idle (16 ms for the 64 x 64 layer, 20 us in 512 chunks of
// these tiles, most of it load latency), and a sum of chunk sums rounds less than one running sum.
__global__ void __launch_bounds__(256)
k_wgrad(const float * __restrict__ A, const float * __restrict__ dY, float * __restrict__ part, uint64_t stride,
		size_t o_w, size_t o_b, uint32_t n, uint32_t a, uint32_t b, uint32_t per) {
	__shared__ float s_a[16][68], s_d[16][68];
	const uint32_t tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
	const uint32_t k0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
	const uint32_t r0 = blockIdx.z * per, r1 = min(n, r0 + per);
	float * out = part + (size_t)blockIdx.z * stride;
	float acc[4][4] = {}, db[4] = {};
	float la[4], ld[4];   // the next 16 rows, loaded while these are multiplied
	auto load = [&](uint32_t rb) {
#pragma unroll
		for (int e = 0; e < 4; ++e) {
			const uint32_t r = rb + ((tid + e * 256) >> 6), c = tid & 63;
			la[e] = r < r1 && k0 + c < a ? A[(size_t)r * a + k0 + c] : 0.f;
			ld[e] = r < r1 && c0 + c < b ? dY[(size_t)r * b + c0 + c] : 0.f;
		}
	};
	load(r0);
	for (uint32_t rb = r0; rb < r1; rb += 16) {
#pragma unroll
		for (int e = 0; e < 4; ++e) {
			const uint32_t r = (tid + e * 256) >> 6, c = tid & 63;
			s_a[r][c] = la[e];
			s_d[r][c] = ld[e];
		}
		__syncthreads();
		if (rb + 16 < r1) load(rb + 16);
		auto row = [&](uint32_t r) {
			const float4 x = *reinterpret_cast<const float4 *>(&s_a[r][ty * 4]);
			const float4 d = *reinterpret_cast<const float4 *>(&s_d[r][tx * 4]);
			const float xs[4] = {x.x, x.y, x.z, x.w}, ds[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
			for (int j = 0; j < 4; ++j) {
				db[j] += ds[j];
#pragma unroll
				for (int i = 0; i < 4; ++i) acc[i][j] = fmaf(xs[i], ds[j], acc[i][j]);
			}
		};
		if (rb + 16 <= r1) {
#pragma unroll
			for (uint32_t r = 0; r < 16; ++r) row(r);
		} else {
			for (uint32_t r = 0; r < r1 - rb; ++r) row(r);
		}
		if (rb + 16 < r1) __syncthreads();
	}
#pragma unroll
	for (int j = 0; j < 4; ++j) {
		const uint32_t c = c0 + tx * 4 + j;
		if (c >= b) break;
		if (k0 == 0 && ty == 0) out[o_b + c] = db[j];
#pragma unroll
		for (int i = 0; i < 4; ++i) {
			const uint32_t k = k0 + ty * 4 + i;
			if (k < a) out[o_w + (size_t)k * b + c] = acc[i][j];
		}
	}
}

// g = sum of the chunks' gradient vectors; a workgroup takes 64 parameters,
// its four waves a quarter of the chunks each.
__global__ void __launch_bounds__(256)
k_sum_chunks(const float * __restrict__ part, uint64_t np, uint32_t chunks, float * __restrict__ g) {
	__shared__ float s[4][64];
	const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	const uint64_t i = (uint64_t)blockIdx.x * 64 + lane;
	float acc = 0.f;
	if (i < np) {
#pragma unroll 8
		for (uint32_t c = chunks * w / 4; c < chunks * (w + 1) / 4; ++c) acc += part[(size_t)c * np + i];
	}
	s[w][lane] = acc;
	__syncthreads();
	if (w == 0 && i < np) g[i] = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
}

__global__ void __launch_bounds__(256)
k_adam(float * __restrict__ p, const float * __restrict__ g, float * __restrict__ m, float * __restrict__ v,
	   uint64_t n, float lr, float b1c, float b2c) {
	const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
	if (i >= n) return;
	const float gi = g[i];
	const float mi = 0.9f * m[i] + 0.1f * gi;
	const float vi = 0.999f * v[i] + 0.001f * gi * gi;
	m[i] = mi;
	v[i] = vi;
	p[i] -= lr * (mi / b1c) / (sqrtf(vi / b2c) + 1e-8f);
}

__global__ void __launch_bounds__(256)
k_gather_rows(const float * __restrict__ src, const uint32_t * __restrict__ idx, float * __restrict__ dst,
			  uint32_t n, uint32_t w) {
	const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
	if (i >= (uint64_t)n * w) return;
	const uint32_t r = (uint32_t)(i / w), c = (uint32_t)(i % w);
	dst[i] = src[(size_t)idx[r] * w + c];
}

uint32_t grid(uint64_t n) { return (uint32_t)std::max<uint64_t>(1, (n + 255) / 256); }

int ensure_batch(tm_mlp * m, uint32_t n) {
	if (n <= m->cap) return TM_OK;
	m->free_batch();
	TM_CHECK(dalloc(&m->d_x, (size_t)n * m->n_in));
	TM_CHECK(dalloc(&m->d_t, (size_t)n * m->n_out));
	TM_CHECK(dalloc(&m->d_h1, (size_t)n * m->h));
	TM_CHECK(dalloc(&m->d_h2, (size_t)n * m->h));
	TM_CHECK(dalloc(&m->d_y, (size_t)n * m->n_out));
	TM_CHECK(dalloc(&m->d_dy, (size_t)n * m->n_out));
	TM_CHECK(dalloc(&m->d_dh1, (size_t)n * m->h));
	TM_CHECK(dalloc(&m->d_dh2, (size_t)n * m->h));
	m->cap = n;
	return TM_OK;
}

dim3 layer_grid(uint32_t n, uint32_t m) { return dim3((n + 63) / 64, (m + 63) / 64); }

// forward on the n rows already in d_x
void forward(tm_mlp * m, uint32_t n) {
	const float * P = m->d_p;
	const float * none = nullptr;
	hipLaunchKernelGGL(k_layer<false>, layer_grid(n, m->h), dim3(256), 0, m->s, m->d_x, P + m->o_w1(), P + m->o_b1(),
					   none, m->d_h1, n, m->n_in, m->h, 1);
	hipLaunchKernelGGL(k_layer<false>, layer_grid(n, m->h), dim3(256), 0, m->s, m->d_h1, P + m->o_w2(), P + m->o_b2(),
					   none, m->d_h2, n, m->h, m->h, 1);
	hipLaunchKernelGGL(k_layer<false>, layer_grid(n, m->n_out), dim3(256), 0, m->s, m->d_h2, P + m->o_w3(),
					   P + m->o_b3(), none, m->d_y, n, m->h, m->n_out, 0);
}

// Row chunks of the weight gradients: up to 512 of at least 32 rows, as far
// as their gradient vectors fit 64 MB.
uint32_t grad_rows(const tm_mlp * m, uint32_t n) {
	const uint64_t most = std::max<uint64_t>(1, std::min<uint64_t>(512, (16ull << 20) / m->n_params));
	return (uint32_t)std::max<uint64_t>(32, (n + most - 1) / most);
}

int ensure_chunks(tm_mlp * m, uint32_t n) {
	const uint32_t per = grad_rows(m, n);
	const uint64_t need = (uint64_t)((n + per - 1) / per) * m->n_params;
	if (need <= m->part_cap) return TM_OK;
	dfree(m->d_part);
	m->part_cap = 0;
	TM_CHECK(dalloc(&m->d_part, need));
	m->part_cap = need;
	return TM_OK;
}

// loss and gradients of the n rows in d_x / d_t; loss left in d_loss
void backward(tm_mlp * m, uint32_t n) {
	const float * P = m->d_p;
	const float * none = nullptr;
	const uint32_t per = grad_rows(m, n), chunks = (n + per - 1) / per;
	const uint64_t np = m->n_params;
	float * part = chunks == 1 ? m->d_g : m->d_part;
	const uint64_t no = (uint64_t)n * m->n_out;
	if (grid(no) > 1) fill_u32(reinterpret_cast<uint32_t *>(m->d_loss), 0, 1, m->s);
	hipLaunchKernelGGL(k_mse, dim3(grid(no)), dim3(256), 0, m->s, m->d_y, m->d_t, m->d_dy, no, m->d_loss);
	hipLaunchKernelGGL(k_wgrad, dim3((m->h + 63) / 64, (m->n_out + 63) / 64, chunks), dim3(256), 0, m->s, m->d_h2,
					   m->d_dy, part, np, m->o_w3(), m->o_b3(), n, m->h, m->n_out, per);
	hipLaunchKernelGGL(k_layer<true>, layer_grid(n, m->h), dim3(256), 0, m->s, m->d_dy, P + m->o_w3(), none, m->d_h2,
					   m->d_dh2, n, m->n_out, m->h, 0);
	hipLaunchKernelGGL(k_wgrad, dim3((m->h + 63) / 64, (m->h + 63) / 64, chunks), dim3(256), 0, m->s, m->d_h1,
					   m->d_dh2, part, np, m->o_w2(), m->o_b2(), n, m->h, m->h, per);
	hipLaunchKernelGGL(k_layer<true>, layer_grid(n, m->h), dim3(256), 0, m->s, m->d_dh2, P + m->o_w2(), none, m->d_h1,
					   m->d_dh1, n, m->h, m->h, 0);
	hipLaunchKernelGGL(k_wgrad, dim3((m->n_in + 63) / 64, (m->h + 63) / 64, chunks), dim3(256), 0, m->s, m->d_x,
					   m->d_dh1, part, np, m->o_w1(), m->o_b1(), n, m->n_in, m->h, per);
	if (chunks > 1)
		hipLaunchKernelGGL(k_sum_chunks, dim3((uint32_t)((np + 63) / 64)), dim3(256), 0, m->s, m->d_part, np, chunks,
						   m->d_g);
}


// ------------------------------------------------------------- unit features

// Reduce the per-lane contribution (sel, c = query popcount, o = popcount of
// query AND partition OR) over the workgroup and, in thread 0, write the
// feature row.  `red` holds NW x 12 words of LDS; two calls in a row must
// use different `red` buffers (the caller alternates two).
template <int NW>
__device__ void unit_row(bool sel, uint32_t c, uint32_t o, const uint32_t * __restrict__ pinfo,
						 const uint32_t * __restrict__ pstat, uint32_t * red, float * __restrict__ row) {
	const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const uint64_t m = __ballot(sel);
	uint32_t sc = sel ? c : 0, sc2 = sel ? c * c : 0, so = sel ? o : 0;
	uint32_t cmin = sel ? c : 0xFFFFFFFFu, cmax = sel ? c : 0, omax = sel ? o : 0;
#pragma unroll
	for (int d = 32; d > 0; d >>= 1) {
		sc += __shfl_xor(sc, d, 64);
		sc2 += __shfl_xor(sc2, d, 64);
		so += __shfl_xor(so, d, 64);
		cmin = min(cmin, (uint32_t)__shfl_xor(cmin, d, 64));
		cmax = max(cmax, (uint32_t)__shfl_xor(cmax, d, 64));
		omax = max(omax, (uint32_t)__shfl_xor(omax, d, 64));
	}
	const uint32_t b0 = (uint32_t)__popcll(__ballot(sel && c < 80));
	const uint32_t b1 = (uint32_t)__popcll(__ballot(sel && c >= 80 && c < 110));
	const uint32_t b2 = (uint32_t)__popcll(__ballot(sel && c >= 110 && c < 140));
	const uint32_t b3 = (uint32_t)__popcll(__ballot(sel && c >= 140));
	if (lane == 0) {
		uint32_t * r = red + wave * 12;
		r[0] = (uint32_t)__popcll(m); r[1] = sc; r[2] = sc2; r[3] = so;
		r[4] = cmin; r[5] = cmax; r[6] = omax;
		r[7] = b0; r[8] = b1; r[9] = b2; r[10] = b3;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		uint32_t n = 0, tsc = 0, tso = 0, tmin = 0xFFFFFFFFu, tmax = 0, tomax = 0, band[4] = {0, 0, 0, 0};
		uint64_t tsc2 = 0;
		for (int w = 0; w < NW; ++w) {
			const uint32_t * r = red + w * 12;
			n += r[0]; tsc += r[1]; tsc2 += r[2]; tso += r[3];
			tmin = min(tmin, r[4]); tmax = max(tmax, r[5]); tomax = max(tomax, r[6]);
			for (int k = 0; k < 4; ++k) band[k] += r[7 + k];
		}
		const float np = (float)pstat[6];
		uint32_t mpop = 0, opop = 0;
		for (int j = 0; j < 6; ++j) {
			mpop += __popc(pinfo[j]);
			opop += __popc(pstat[j]);
		}
		float f[N_FEAT];
		for (int k = 0; k < N_FEAT; ++k) f[k] = 0.f;
		f[0] = log2f(1.f + np) / 20.f;
		f[1] = (float)mpop / 64.f;
		f[11] = np > 0.f ? (float)pstat[7] / np / 64.f : 0.f;
		f[12] = (float)opop / 192.f;
		if (n && np > 0.f) {   // a partition without filters is no work
			const float inv = 1.f / (float)n;
			const float mean = (float)tsc * inv;
			const float var = fmaxf((float)tsc2 * inv - mean * mean, 0.f);
			f[2] = log2f(1.f + (float)n) / 12.f;
			f[3] = mean / 192.f;
			f[4] = sqrtf(var) / 192.f;
			f[5] = (float)tmin / 192.f;
			f[6] = (float)tmax / 192.f;
			for (int k = 0; k < 4; ++k) f[7 + k] = (float)band[k] * inv;
			f[13] = (float)tso * inv / 192.f;
			f[14] = (float)tomax / 192.f;
			f[15] = log2f(1.f + (float)n * np) / 32.f;
		}
		for (int k = 0; k < N_FEAT; ++k) row[k] = f[k];
	}
}

__device__ inline uint32_t pop6(const uint32_t * w) {
	return __popc(w[0]) + __popc(w[1]) + __popc(w[2]) + __popc(w[3]) + __popc(w[4]) + __popc(w[5]);
}

// One 256-thread workgroup per plain unit.
__global__ void __launch_bounds__(256)
k_unit_features_plain(dev_fib_view f, const uint32_t * __restrict__ q, const uint32_t * __restrict__ list,
					  const uint4 * __restrict__ units, float * __restrict__ out) {
	__shared__ uint32_t red[2][4 * 12];
	const uint4 u = units[blockIdx.x];
	const uint32_t p = u.x;
	const uint32_t * pinfo = f.part_info + (size_t)p * 8;
	const uint32_t * pstat = f.part_stat + (size_t)p * 8;
	// batches hold at most 256 queries: thread t takes query t
	uint32_t c = 0, o = 0;
	bool any = false;
	const uint32_t t = threadIdx.x;
	if (t < u.z) {
		const uint32_t qi = list[u.w + t];
		const uint32_t * w = q + (size_t)qi * 8;
		c = pop6(w);
		o = __popc(w[0] & pstat[0]) + __popc(w[1] & pstat[1]) + __popc(w[2] & pstat[2]) +
			__popc(w[3] & pstat[3]) + __popc(w[4] & pstat[4]) + __popc(w[5] & pstat[5]);
		any = true;
	}
	unit_row<4>(any, c, o, pinfo, pstat, red[0], out + (size_t)blockIdx.x * N_FEAT);
}

// One workgroup per query tile (NQT <= 256 queries, one per thread); loops
// over the partitions.
__global__ void __launch_bounds__(256)
k_unit_features_tiles(dev_fib_view f, const uint32_t * __restrict__ q, uint32_t nq, uint32_t nqt,
					  float * __restrict__ out) {
	__shared__ uint32_t red[2][4 * 12];
	const uint32_t t = blockIdx.x, P = f.n_parts;
	const uint32_t qi = t * nqt + threadIdx.x;
	const bool valid = threadIdx.x < nqt && qi < nq;
	uint32_t w[6] = {0, 0, 0, 0, 0, 0};
	if (valid)
		for (int j = 0; j < 6; ++j) w[j] = q[(size_t)qi * 8 + j];
	const uint32_t c = pop6(w);
	for (uint32_t p = 0; p < P; ++p) {
		const uint32_t * pinfo = f.part_info + (size_t)p * 8;
		const uint32_t * pstat = f.part_stat + (size_t)p * 8;
		bool sel = valid;
		uint32_t o = 0;
		for (int j = 0; j < 6; ++j) {
			sel = sel && (pinfo[j] & ~w[j]) == 0;
			o += __popc(w[j] & pstat[j]);
		}
		unit_row<4>(sel, c, o, pinfo, pstat, red[p & 1], out + ((size_t)t * P + p) * N_FEAT);
	}
}

// ------------------------------------------------------------- fused inference

// One thread per row of the IN-H-H-OUT network; parameters staged in LDS
// and read as broadcasts.
template <int IN, int H, int OUT>
__global__ void __launch_bounds__(256)
k_mlp_fused(const float * __restrict__ P, const float * __restrict__ X, uint32_t n, float * __restrict__ Y) {
	constexpr int NP = IN * H + H + H * H + H + H * OUT + OUT;
	__shared__ float4 s_p4[(NP + 3) / 4];
	float * s_p = reinterpret_cast<float *>(s_p4);
	for (int i = threadIdx.x; i < NP; i += 256) s_p[i] = P[i];
	__syncthreads();
	const uint32_t r = blockIdx.x * 256 + threadIdx.x;
	if (r >= n) return;
	const float * W1 = s_p, * B1 = W1 + IN * H, * W2 = B1 + H, * B2 = W2 + H * H, * W3 = B2 + H, * B3 = W3 + H * OUT;
	float x[IN];
#pragma unroll
	for (int k = 0; k < IN; ++k) x[k] = X[(size_t)r * IN + k];
	float h1[H];
#pragma unroll
	for (int j = 0; j < H; ++j) h1[j] = B1[j];
#pragma unroll
	for (int k = 0; k < IN; ++k)
#pragma unroll
		for (int j = 0; j < H; ++j) h1[j] = fmaf(x[k], W1[k * H + j], h1[j]);
#pragma unroll
	for (int j = 0; j < H; ++j) h1[j] = fmaxf(h1[j], 0.f);
	float y[OUT];
#pragma unroll
	for (int o = 0; o < OUT; ++o) y[o] = B3[o];
	for (int j = 0; j < H; j += 4) {
		float a0 = B2[j], a1 = B2[j + 1], a2 = B2[j + 2], a3 = B2[j + 3];
#pragma unroll
		for (int k = 0; k < H; ++k) {
			const float4 w = *reinterpret_cast<const float4 *>(&W2[k * H + j]);
			a0 = fmaf(h1[k], w.x, a0);
			a1 = fmaf(h1[k], w.y, a1);
			a2 = fmaf(h1[k], w.z, a2);
			a3 = fmaf(h1[k], w.w, a3);
		}
		a0 = fmaxf(a0, 0.f); a1 = fmaxf(a1, 0.f); a2 = fmaxf(a2, 0.f); a3 = fmaxf(a3, 0.f);
#pragma unroll
		for (int o = 0; o < OUT; ++o)
			y[o] = fmaf(a0, W3[j * OUT + o],
						fmaf(a1, W3[(j + 1) * OUT + o], fmaf(a2, W3[(j + 2) * OUT + o], fmaf(a3, W3[(j + 3) * OUT + o], y[o]))));
	}
#pragma unroll
	for (int o = 0; o < OUT; ++o) Y[(size_t)r * OUT + o] = y[o];
}

// One thread per tile: decoded sums over its partitions.
__global__ void __launch_bounds__(256)
k_tile_costs(const float * __restrict__ X, const float * __restrict__ Y, uint32_t n_tiles, uint32_t P,
			 float * __restrict__ cost, float * __restrict__ hits, float * __restrict__ keys) {
	const uint32_t t = blockIdx.x * 256 + threadIdx.x;
	if (t >= n_tiles) return;
	float c = 0.f, h = 0.f, k = 0.f;
	for (uint32_t p = 0; p < P; ++p) {
		const size_t r = (size_t)t * P + p;
		if (X[r * N_FEAT + 2] <= 0.f) continue;   // no query of the tile selects p
		h += exp2f(16.f * fmaxf(Y[r * N_TARGET], 0.f)) - 1.f;
		k += exp2f(16.f * fmaxf(Y[r * N_TARGET + 1], 0.f)) - 1.f;
		c += exp2f(16.f * fmaxf(Y[r * N_TARGET + 2], 0.f)) - 1.f;
	}
	cost[t] = c;
	hits[t] = h;
	keys[t] = k;
}

} // namespace

namespace tmx {

void launch_unit_features_plain(const dev_fib_view & f, const uint32_t * q, const uint32_t * list,
								const uint4 * units, uint32_t n_units, float * out, hipStream_t s) {
	if (n_units == 0) return;
	hipLaunchKernelGGL(k_unit_features_plain, dim3(n_units), dim3(256), 0, s, f, q, list, units, out);
}

void launch_unit_features_tiles(const dev_fib_view & f, const uint32_t * q, uint32_t nq, uint32_t nqt,
								uint32_t n_tiles, float * out, hipStream_t s) {
	if (n_tiles == 0 || f.n_parts == 0) return;
	hipLaunchKernelGGL(k_unit_features_tiles, dim3(n_tiles), dim3(256), 0, s, f, q, nq, nqt, out);
}

bool mlp_fused_shape(const tm_mlp * m) {
	return m && m->n_in == N_FEAT && m->h == 64 && m->n_out == N_TARGET;
}

int mlp_infer(const tm_mlp * m, const float * x, uint32_t n, float * y, hipStream_t s) {
	if (!mlp_fused_shape(m)) return set_error(TM_ERR_INVALID, "cost model must be %d-64-64-%d", N_FEAT, N_TARGET);
	if (n == 0) return TM_OK;
	hipLaunchKernelGGL((k_mlp_fused<N_FEAT, 64, N_TARGET>), dim3((n + 255) / 256), dim3(256), 0, s, m->d_p, x, n, y);
	return TM_OK;
}

void launch_tile_costs(const float * x, const float * y, uint32_t n_tiles, uint32_t P, float * cost, float * hits,
					   float * keys, hipStream_t s) {
	if (n_tiles == 0) return;
	hipLaunchKernelGGL(k_tile_costs, dim3((n_tiles + 255) / 256), dim3(256), 0, s, x, y, n_tiles, P, cost, hits, keys);
}

} // namespace tmx

extern "C" {

int tm_mlp_create(uint32_t n_in, uint32_t n_hidden, uint32_t n_out, uint64_t seed, tm_mlp ** out) {
	if (!out || n_in == 0 || n_hidden == 0 || n_out == 0 || n_in > 4096 || n_hidden > 4096 || n_out > 4096)
		return set_error(TM_ERR_INVALID, "bad MLP shape");
	TM_CHECK(require_device());
	tm_mlp * m = new tm_mlp();
	m->n_in = n_in;
	m->h = n_hidden;
	m->n_out = n_out;
	m->n_params = (uint64_t)n_in * n_hidden + n_hidden + (uint64_t)n_hidden * n_hidden + n_hidden +
				  (uint64_t)n_hidden * n_out + n_out;
	int rc = dalloc(&m->d_p, m->n_params);
	if (rc == TM_OK) rc = dalloc(&m->d_g, m->n_params);
	if (rc == TM_OK) rc = dalloc(&m->d_m, m->n_params);
	if (rc == TM_OK) rc = dalloc(&m->d_v, m->n_params);
	if (rc == TM_OK) rc = dalloc(&m->d_loss, 1);
	if (rc == TM_OK && hipStreamCreateWithFlags(&m->s, hipStreamNonBlocking) != hipSuccess)
		rc = set_error(TM_ERR_HIP, "hipStreamCreate failed");
	if (rc != TM_OK) {
		m->release();
		delete m;
		return rc;
	}
	// He initialisation, deterministic in the seed
	std::vector<float> p(m->n_params, 0.f);
	std::mt19937_64 rng(seed);
	auto init = [&](size_t off, uint32_t fan_in, uint64_t count) {
		std::normal_distribution<float> nd(0.f, std::sqrt(2.f / (float)fan_in));
		for (uint64_t i = 0; i < count; ++i) p[off + i] = nd(rng);
	};
	init(m->o_w1(), n_in, (uint64_t)n_in * n_hidden);
	init(m->o_w2(), n_hidden, (uint64_t)n_hidden * n_hidden);
	init(m->o_w3(), n_hidden, (uint64_t)n_hidden * n_out);
	std::vector<float> zero(m->n_params, 0.f);
	if (hipMemcpy(m->d_p, p.data(), m->n_params * 4, hipMemcpyHostToDevice) != hipSuccess ||
		hipMemcpy(m->d_m, zero.data(), m->n_params * 4, hipMemcpyHostToDevice) != hipSuccess ||
		hipMemcpy(m->d_v, zero.data(), m->n_params * 4, hipMemcpyHostToDevice) != hipSuccess) {
		m->release();
		delete m;
		return set_error(TM_ERR_HIP, "MLP parameter upload failed");
	}
	*out = m;
	return TM_OK;
}

int tm_mlp_destroy(tm_mlp * m) {
	if (!m) return TM_OK;
	if (dev().device >= 0) (void)hipSetDevice(dev().device);
	m->release();
	delete m;
	return TM_OK;
}

uint64_t tm_mlp_param_count(const tm_mlp * m) { return m ? m->n_params : 0; }

int tm_mlp_get_params(const tm_mlp * m, float * params, uint64_t n) {
	if (!m || !params || n != m->n_params) return set_error(TM_ERR_INVALID, "bad parameter buffer");
	TM_CHECK(require_device());
	TM_HIP(hipMemcpy(params, m->d_p, n * 4, hipMemcpyDeviceToHost));
	return TM_OK;
}

int tm_mlp_set_params(tm_mlp * m, const float * params, uint64_t n) {
	if (!m || !params || n != m->n_params) return set_error(TM_ERR_INVALID, "bad parameter buffer");
	TM_CHECK(require_device());
	TM_HIP(hipMemcpy(m->d_p, params, n * 4, hipMemcpyHostToDevice));
	return TM_OK;
}

int tm_mlp_forward(tm_mlp * m, const float * x, uint32_t n, float * y) {
	if (!m || (n && (!x || !y))) return set_error(TM_ERR_INVALID, "NULL argument");
	if (n == 0) return TM_OK;
	TM_CHECK(require_device());
	TM_CHECK(ensure_batch(m, n));
	TM_HIP(hipMemcpyAsync(m->d_x, x, (size_t)n * m->n_in * 4, hipMemcpyHostToDevice, m->s));
	if (tmx::mlp_fused_shape(m))   // the kernel the scheduler prices with
		TM_CHECK(tmx::mlp_infer(m, m->d_x, n, m->d_y, m->s));
	else
		forward(m, n);
	TM_HIP(hipGetLastError());
	TM_HIP(hipMemcpyAsync(y, m->d_y, (size_t)n * m->n_out * 4, hipMemcpyDeviceToHost, m->s));
	TM_HIP(hipStreamSynchronize(m->s));
	return TM_OK;
}

int tm_mlp_loss_grad(tm_mlp * m, const float * x, const float * t, uint32_t n, float * loss, float * grad) {
	if (!m || !x || !t || n == 0) return set_error(TM_ERR_INVALID, "bad argument");
	TM_CHECK(require_device());
	TM_CHECK(ensure_batch(m, n));
	TM_CHECK(ensure_chunks(m, n));
	TM_HIP(hipMemcpyAsync(m->d_x, x, (size_t)n * m->n_in * 4, hipMemcpyHostToDevice, m->s));
	TM_HIP(hipMemcpyAsync(m->d_t, t, (size_t)n * m->n_out * 4, hipMemcpyHostToDevice, m->s));
	forward(m, n);
	backward(m, n);
	TM_HIP(hipGetLastError());
	float l = 0.f;
	TM_HIP(hipMemcpyAsync(&l, m->d_loss, 4, hipMemcpyDeviceToHost, m->s));
	if (grad) TM_HIP(hipMemcpyAsync(grad, m->d_g, m->n_params * 4, hipMemcpyDeviceToHost, m->s));
	TM_HIP(hipStreamSynchronize(m->s));
	if (loss) *loss = l;
	return TM_OK;
}

int tm_mlp_train(tm_mlp * m, const float * x, const float * t, uint32_t n, uint32_t epochs, uint32_t batch,
				 float lr, uint64_t seed, float * loss) {
	if (!m || !x || !t || n == 0 || batch == 0 || epochs == 0) return set_error(TM_ERR_INVALID, "bad argument");
	TM_CHECK(require_device());
	const uint32_t bs = std::min(batch, n);
	TM_CHECK(ensure_batch(m, bs));
	TM_CHECK(ensure_chunks(m, bs));
	if (n % bs) TM_CHECK(ensure_chunks(m, n % bs));   // the last batch's chunks may be more
	float * dX = nullptr, * dT = nullptr;
	uint32_t * dIdx = nullptr;
	TM_CHECK(dalloc(&dX, (size_t)n * m->n_in));
	int rc = dalloc(&dT, (size_t)n * m->n_out);
	if (rc == TM_OK) rc = dalloc(&dIdx, n);
	std::vector<uint32_t> idx(n);
	for (uint32_t i = 0; i < n; ++i) idx[i] = i;
	std::mt19937_64 rng(seed);
	float last = 0.f;
	if (rc == TM_OK && (hipMemcpyAsync(dX, x, (size_t)n * m->n_in * 4, hipMemcpyHostToDevice, m->s) != hipSuccess ||
						hipMemcpyAsync(dT, t, (size_t)n * m->n_out * 4, hipMemcpyHostToDevice, m->s) != hipSuccess))
		rc = set_error(TM_ERR_HIP, "training data upload failed");
	for (uint32_t e = 0; e < epochs && rc == TM_OK; ++e) {
		std::shuffle(idx.begin(), idx.end(), rng);
		if (hipMemcpyAsync(dIdx, idx.data(), (size_t)n * 4, hipMemcpyHostToDevice, m->s) != hipSuccess) {
			rc = set_error(TM_ERR_HIP, "index upload failed");
			break;
		}
		double esum = 0.0;
		uint32_t nb = 0;
		for (uint32_t b0 = 0; b0 < n; b0 += bs) {
			const uint32_t cnt = std::min(bs, n - b0);
			hipLaunchKernelGGL(k_gather_rows, dim3(grid((uint64_t)cnt * m->n_in)), dim3(256), 0, m->s, dX, dIdx + b0,
							   m->d_x, cnt, m->n_in);
			hipLaunchKernelGGL(k_gather_rows, dim3(grid((uint64_t)cnt * m->n_out)), dim3(256), 0, m->s, dT,
							   dIdx + b0, m->d_t, cnt, m->n_out);
			forward(m, cnt);
			backward(m, cnt);
			++m->step;
			const float b1c = 1.f - std::pow(0.9f, (float)m->step), b2c = 1.f - std::pow(0.999f, (float)m->step);
			hipLaunchKernelGGL(k_adam, dim3(grid(m->n_params)), dim3(256), 0, m->s, m->d_p, m->d_g, m->d_m, m->d_v,
							   m->n_params, lr, b1c, b2c);
			if (e + 1 == epochs) {
				float l = 0.f;
				if (hipMemcpyAsync(&l, m->d_loss, 4, hipMemcpyDeviceToHost, m->s) != hipSuccess ||
					hipStreamSynchronize(m->s) != hipSuccess) {
					rc = set_error(TM_ERR_HIP, "loss readback failed");
					break;
				}
				esum += l;
				++nb;
			}
		}
		if (hipGetLastError() != hipSuccess && rc == TM_OK) rc = set_error(TM_ERR_HIP, "training kernel failed");
		if (nb) last = (float)(esum / nb);
	}
	if (rc == TM_OK && hipStreamSynchronize(m->s) != hipSuccess) rc = set_error(TM_ERR_HIP, "training sync failed");
	dfree(dX);
	dfree(dT);
	dfree(dIdx);
	if (loss) *loss = last;
	return rc;
}

} // extern "C"
