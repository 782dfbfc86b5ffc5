// k_volume.hip -- volume stages of meshify() on gfx950.
//
//  * pre-smooth (src/meshify.c:170-216) fused with the intensity range scan
//    (src/meshify.c:306-311) and a speculative threshold mask;
//  * threshold mask as packed bits (src/meshify.c:325-330);
//  * one-voxel dilation of a bit mask (src/meshify.c:218-264);
//  * fill/outside/edge-darken apply with bounding box (src/meshify.c:332-371);
//  * histograms of setThreshold() (src/isolevel.c:35-139, 245-262).
//
// Bit volumes: one uint32 word per 32 voxels of an x-row, W = ceil(nx/32)
// words per row, word index wx + W*(y + ny*z), bit b <-> x = 32*wx + b.
#include <float.h>

#include "n2m_device.cuh"
#include "n2m_internal.h"

namespace n2m {

// ---------------------------------------------------------------------------
// Pre-smooth.  2.5-D streaming: a workgroup owns a 64x8 column tile and a
// z-chunk; per input plane it stages the tile plus a 2-voxel halo in LDS,
// applies the x pass then the y pass (each rounded to float, as the
// reference stores between passes), and keeps the last five x/y-smoothed
// planes per column in registers for the z pass.  Every pass computes
// float*double products summed left to right in double (meshify.c:189).
// ---------------------------------------------------------------------------
constexpr int SM_TX = 64, SM_TY = 8, SM_ZC = 32, SM_BS = 256; // 2 columns per thread

__device__ __forceinline__ float tap5(float a, float b, float c, float d, float e)
{
	const double w0 = 0.45, w1 = 0.225, w2 = 0.05;
	double acc = a * w2;
	acc = acc + b * w1;
	acc = acc + c * w0;
	acc = acc + d * w1;
	acc = acc + e * w2;
	return (float)acc;
}

// Isolevels whose threshold masks the smoothing writes as it goes: mask k
// (out >= v[k]) goes to bits + k * nwords.
struct IsoMasks {
	float v[N2M_SMOOTH_MASKS];
	int n;
	size_t nwords;
};

// Smooth the TX x TY tile (x0, y0, [z0, z1)) of an nx*ny*nz volume read
// through `src(x, y, z)` (only called inside the volume) into out; returns
// the tile's min/max through lmin/lmax (per thread) and, for TX = 64 (one
// wave per tile row), writes speculative mask bits for the isolevels of
// `iso` when bits != null.
template <int TX, int TY, class Src>
__device__ __forceinline__ void smooth_tile(const Src &src, float *__restrict__ out, int nx, int ny, int nz,
                                            int x0, int y0, int z0, int z1, const IsoMasks &iso,
                                            uint32_t *__restrict__ bits, int W, float &lmin, float &lmax)
{
	constexpr int CPT = TX * TY / SM_BS, RPP = SM_BS / TX; // columns per thread, rows per pass
	static_assert(CPT * SM_BS == TX * TY && RPP * TX == SM_BS, "tile must tile the workgroup");
	__shared__ float s_in[TY + 4][TX + 4];
	__shared__ float s_x[TY + 4][TX];
	const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
	const size_t nxy = (size_t)nx * ny;
	float ring[CPT][5];
#pragma unroll
	for (int c = 0; c < CPT; c++)
#pragma unroll
		for (int k = 0; k < 5; k++)
			ring[c][k] = 0.f;
	const int x = x0 + tx;
	// the plane's halo tile is loaded into registers one plane ahead, so its
	// memory latency overlaps the previous plane's passes
	constexpr int NIN = (TY + 4) * (TX + 4), NL = (NIN + SM_BS - 1) / SM_BS;
	float pre[NL];
	auto fetch = [&](int zz) {
#pragma unroll
		for (int q = 0; q < NL; q++) {
			const int i = q * SM_BS + threadIdx.x;
			const int ly = i / (TX + 4), lx = i % (TX + 4);
			const int gx = x0 - 2 + lx, gy = y0 - 2 + ly;
			float v = 0.f;
			if (i < NIN && zz >= 0 && zz < nz && gx >= 0 && gx < nx && gy >= 0 && gy < ny)
				v = src(gx, gy, zz);
			pre[q] = v;
		}
	};
	fetch(z0 - 2);
	for (int zz = z0 - 2; zz <= z1 + 1; zz++) {
		const bool have = zz >= 0 && zz < nz;
		if (have) {
#pragma unroll
			for (int q = 0; q < NL; q++) {
				const int i = q * SM_BS + threadIdx.x;
				if (i < NIN)
					s_in[i / (TX + 4)][i % (TX + 4)] = pre[q];
			}
		}
		if (zz + 1 <= z1 + 1)
			fetch(zz + 1);
		if (have) {
			__syncthreads();
			for (int i = threadIdx.x; i < (TY + 4) * TX; i += SM_BS) {
				int ly = i / TX, lx = i % TX;
				int gx = x0 + lx;
				float v;
				if (gx >= 2 && gx < nx - 2)
					v = tap5(s_in[ly][lx], s_in[ly][lx + 1], s_in[ly][lx + 2], s_in[ly][lx + 3],
					         s_in[ly][lx + 4]);
				else
					v = s_in[ly][lx + 2];
				s_x[ly][lx] = v;
			}
			__syncthreads();
		}
#pragma unroll
		for (int c = 0; c < CPT; c++) {
			const int ly = ty + c * RPP;
			const int y = y0 + ly;
			float v = 0.f;
			if (have) {
				if (y >= 2 && y < ny - 2)
					v = tap5(s_x[ly][tx], s_x[ly + 1][tx], s_x[ly + 2][tx], s_x[ly + 3][tx],
					         s_x[ly + 4][tx]);
				else
					v = s_x[ly + 2][tx];
			}
			ring[c][0] = ring[c][1];
			ring[c][1] = ring[c][2];
			ring[c][2] = ring[c][3];
			ring[c][3] = ring[c][4];
			ring[c][4] = v;
		}
		const int zo = zz - 2;
		if (zo >= z0 && zo < z1) {
#pragma unroll
			for (int c = 0; c < CPT; c++) {
				const int y = y0 + ty + c * RPP;
				float o;
				if (zo >= 2 && zo < nz - 2)
					o = tap5(ring[c][0], ring[c][1], ring[c][2], ring[c][3], ring[c][4]);
				else
					o = ring[c][2];
				const bool valid = x < nx && y < ny;
				if (valid) {
					out[(size_t)zo * nxy + (size_t)y * nx + x] = o;
					lmin = fminf(lmin, o);
					lmax = fmaxf(lmax, o);
				}
				if (TX == 64 && bits) { // speculative threshold masks
					const int wx = x0 / 32;
					const size_t wi = (size_t)wx + (size_t)W * ((size_t)y + (size_t)ny * zo);
					for (int k = 0; k < iso.n; k++) {
						const unsigned long long m = __ballot(valid && o >= iso.v[k]);
						uint32_t *bk = bits + k * iso.nwords;
						if (y < ny) {
							if (tx == 0)
								bk[wi] = (uint32_t)m;
							else if (tx == 32 && wx + 1 < W)
								bk[wi + 1] = (uint32_t)(m >> 32);
						}
					}
				}
			}
		}
		if (have)
			__syncthreads();
	}
}

// block-wide min/max into range[0] (ord min) and range[1] (ord max)
__device__ __forceinline__ void reduce_range(float lmin, float lmax, uint32_t *range)
{
	__shared__ uint32_t s_red[2][SM_BS / N2M_WAVE];
	uint32_t omin = wave_min_u32(f2ord(lmin)), omax = wave_max_u32(f2ord(lmax));
	if (lane_id() == 0) {
		s_red[0][wave_id()] = omin;
		s_red[1][wave_id()] = omax;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		for (int w = 1; w < SM_BS / N2M_WAVE; w++) {
			omin = min(omin, s_red[0][w]);
			omax = max(omax, s_red[1][w]);
		}
		if (omin < ld_agent(&range[0]))
			atomicMin(&range[0], omin);
		if (omax > ld_agent(&range[1]))
			atomicMax(&range[1], omax);
	}
}

struct ImgSrc {
	const float *__restrict__ img;
	int nx;
	size_t nxy;
	__device__ float operator()(int x, int y, int z) const { return img[(size_t)z * nxy + (size_t)y * nx + x]; }
};

__global__ void __launch_bounds__(SM_BS)
k_smooth(const float *__restrict__ in, float *__restrict__ out, int nx, int ny, int nz, int zc,
         uint32_t *__restrict__ range /* [0]=ord min, [1]=ord max */, IsoMasks iso,
         uint32_t *__restrict__ bits, int W)
{
	const int x0 = blockIdx.x * SM_TX, y0 = blockIdx.y * SM_TY;
	const int z0 = blockIdx.z * zc, z1 = min(z0 + zc, nz);
	float lmin = __builtin_inff(), lmax = -__builtin_inff();
	ImgSrc src{in, nx, (size_t)nx * ny};
	smooth_tile<SM_TX, SM_TY>(src, out, nx, ny, nz, x0, y0, z0, z1, iso, bits, W, lmin, lmax);
	reduce_range(lmin, lmax, range);
}

// ---------------------------------------------------------------------------
// Batched atlas (src/nii2mesh.c:492-583).  Each label is processed on its
// own crop (label box grown by 4 voxels, clipped to the volume): beyond 2
// voxels from the label its binarised and smoothed volume is 0, so the crop
// reproduces the full-volume smoothing, range, darkening and bounding box.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int atlas_label_of(float v, int nlabel)
{
	float r = rintf(v); // the only label whose open interval (i-0.5, i+0.5) can hold v
	if (!(r >= 1.0f && r <= (float)nlabel))
		return 0;
	int i = (int)r;
	float lo = (float)((double)i - 0.5), hi = (float)((double)i + 0.5); // src/nii2mesh.c:555-556
	return (v > lo && v < hi) ? i : 0;
}

// per label: voxel count and box (stats[7*i] = count, min xyz, max xyz);
// PRIV: accumulate in LDS (7 * (nlabel + 1) words) and flush once per block.
// Each block reads one contiguous run of voxels, AS_UNROLL loads per thread
// in flight, so it meets few labels and flushes few.  Within a wave the
// voxels are consecutive along x: a run of lanes with one label in one row
// is merged by its first lane (count = run length, x from its two ends, y
// and z shared), one set of atomics per run.  I32: the volume has fewer
// than 2^32 voxels, so coordinates take 32-bit division.
constexpr int AS_UNROLL = 4;

template <bool PRIV, bool I32>
__device__ __forceinline__ void atlas_stats_voxel(int i, size_t v, int nx, int ny, uint32_t *__restrict__ s_st,
                                                  uint32_t *__restrict__ stats)
{
	if (!__ballot(i != 0))
		return;
	uint32_t x, y, z;
	if (I32) {
		const uint32_t w = (uint32_t)v, r = w / (uint32_t)nx;
		x = w - r * (uint32_t)nx;
		y = r % (uint32_t)ny;
		z = r / (uint32_t)ny;
	} else {
		x = (uint32_t)(v % nx);
		y = (uint32_t)((v / nx) % ny);
		z = (uint32_t)(v / ((size_t)nx * ny));
	}
	const int lane = lane_id();
	const int iprev = __shfl_up(i, 1);
	const bool head = lane == 0 || i != iprev || x == 0; // a run starts
	const unsigned long long heads = __ballot(head);
	if (!head || !i)
		return;
	const unsigned long long after = lane == N2M_WAVE - 1 ? 0ull : heads & (~0ull << (lane + 1));
	const uint32_t len = (uint32_t)((after ? __ffsll((long long)after) - 1 : N2M_WAVE) - lane);
	uint32_t *st = PRIV ? s_st + 7 * i : stats + 7 * i;
	atomicAdd(&st[0], len);
	atomicMin(&st[1], x);
	atomicMin(&st[2], y);
	atomicMin(&st[3], z);
	atomicMax(&st[4], x + len - 1);
	atomicMax(&st[5], y);
	atomicMax(&st[6], z);
}

template <bool PRIV, bool I32>
__global__ void __launch_bounds__(256)
k_atlas_stats(const float *__restrict__ labels, int nx, int ny, int nz, int nlabel, uint32_t *__restrict__ stats)
{
	extern __shared__ uint32_t s_st[];
	if (PRIV) {
		for (int i = threadIdx.x; i <= nlabel; i += blockDim.x) {
			s_st[7 * i] = 0;
			s_st[7 * i + 1] = s_st[7 * i + 2] = s_st[7 * i + 3] = 0xffffffffu;
			s_st[7 * i + 4] = s_st[7 * i + 5] = s_st[7 * i + 6] = 0u;
		}
		__syncthreads();
	}
	const size_t n = (size_t)nx * ny * nz;
	constexpr size_t STEP = 256 * AS_UNROLL;
	const size_t per = ((n + gridDim.x - 1) / gridDim.x + STEP - 1) / STEP * STEP;
	const size_t v0 = blockIdx.x * per, v1 = v0 + per < n ? v0 + per : n;
	for (size_t vb = v0; vb < v1; vb += STEP) { // uniform trip count: whole waves take part
		float val[AS_UNROLL];
#pragma unroll
		for (int u = 0; u < AS_UNROLL; u++) {
			const size_t v = vb + u * 256 + threadIdx.x;
			val[u] = v < v1 ? labels[v] : 0.0f;
		}
#pragma unroll
		for (int u = 0; u < AS_UNROLL; u++)
			atlas_stats_voxel<PRIV, I32>(atlas_label_of(val[u], nlabel), vb + u * 256 + threadIdx.x, nx, ny, s_st,
			                             stats);
	}
	if (!PRIV)
		return;
	__syncthreads();
	for (int i = threadIdx.x; i <= nlabel; i += blockDim.x) {
		if (!s_st[7 * i])
			continue;
		atomicAdd(&stats[7 * i], s_st[7 * i]);
		for (int k = 1; k <= 3; k++)
			atomicMin(&stats[7 * i + k], s_st[7 * i + k]);
		for (int k = 4; k <= 6; k++)
			atomicMax(&stats[7 * i + k], s_st[7 * i + k]);
	}
}

void launch_atlas_stats(const float *labels, int nx, int ny, int nz, int nlabel, uint32_t *stats, hipStream_t s)
{
	size_t n = (size_t)nx * ny * nz;
	size_t b = (n + 1023) / 1024;
	b = b > 2048 ? 2048 : (b < 1 ? 1 : b);
	const size_t lds = (size_t)7 * (nlabel + 1) * 4;
	const bool i32 = n <= 0xffffffffull;
	if (nlabel <= 1023 && i32)
		hipLaunchKernelGGL((k_atlas_stats<true, true>), dim3((unsigned)b), dim3(256), lds, s, labels, nx, ny, nz, nlabel,
		                   stats);
	else if (nlabel <= 1023)
		hipLaunchKernelGGL((k_atlas_stats<true, false>), dim3((unsigned)b), dim3(256), lds, s, labels, nx, ny, nz,
		                   nlabel, stats);
	else if (i32)
		hipLaunchKernelGGL((k_atlas_stats<false, true>), dim3((unsigned)b), dim3(256), 0, s, labels, nx, ny, nz, nlabel,
		                   stats);
	else
		hipLaunchKernelGGL((k_atlas_stats<false, false>), dim3((unsigned)b), dim3(256), 0, s, labels, nx, ny, nz,
		                   nlabel, stats);
}

// the binarised label (src/nii2mesh.c:557-563) read inside a task's crop
struct LabelSrc {
	const float *__restrict__ labels;
	int gnx;
	size_t gnxy;
	int ox, oy, oz;
	float lo, hi;
	__device__ float operator()(int x, int y, int z) const
	{
		float v = labels[(size_t)(oz + z) * gnxy + (size_t)(oy + y) * gnx + (ox + x)];
		return (v > lo && v < hi) ? 1.0f : 0.0f;
	}
};

// Crop tile shapes the atlas autotuner chooses from (x, y, z-chunk).
#define N2M_ATLAS_TILES(X) X(0, 64, 8, 32) X(1, 32, 8, 16) X(2, 16, 16, 16) X(3, 32, 8, 32)

// smooth (or just binarise) every task's crop; ranges[2*t] = ord min/max.
// LOOP: persistent, the grid walks the `nwork` items of the block map in
// strides of its own size; otherwise workgroup b takes item b.
template <int TX, int TY, int ZC>
__device__ __forceinline__ void atlas_smooth_item(const float *__restrict__ labels, int gnx, int gny,
                                                  const AtlasTask *__restrict__ tasks,
                                                  const uint32_t *__restrict__ blockTask, unsigned b, int smooth,
                                                  float *__restrict__ crops, uint32_t *__restrict__ ranges)
{
	const int ti = (int)blockTask[b];
	const AtlasTask t = tasks[ti];
	const int local = (int)b - t.first_block;
	LabelSrc src{labels, gnx, (size_t)gnx * gny, t.ox, t.oy, t.oz, t.lo, t.hi};
	float *out = crops + t.off;
	float lmin = __builtin_inff(), lmax = -__builtin_inff();
	if (smooth) {
		const int tx = (t.nx + TX - 1) / TX, ty = (t.ny + TY - 1) / TY;
		const int bx = local % tx, by = (local / tx) % ty, bz = local / (tx * ty);
		const int z0 = bz * ZC, z1 = min(z0 + ZC, t.nz);
		smooth_tile<TX, TY>(src, out, t.nx, t.ny, t.nz, bx * TX, by * TY, z0, z1, IsoMasks{}, nullptr, 0, lmin, lmax);
	} else {
		const size_t n = (size_t)t.nx * t.ny * t.nz;
		const size_t v = (size_t)local * SM_BS + threadIdx.x;
		if (v < n) {
			int x = (int)(v % t.nx), y = (int)((v / t.nx) % t.ny), z = (int)(v / ((size_t)t.nx * t.ny));
			float o = src(x, y, z);
			out[v] = o;
			lmin = o;
			lmax = o;
		}
	}
	reduce_range(lmin, lmax, &ranges[2 * ti]);
}

template <int TX, int TY, int ZC, bool LOOP>
__global__ void __launch_bounds__(SM_BS)
k_atlas_smooth(const float *__restrict__ labels, int gnx, int gny, const AtlasTask *__restrict__ tasks,
               const uint32_t *__restrict__ blockTask, unsigned nwork, int smooth, float *__restrict__ crops,
               uint32_t *__restrict__ ranges)
{
	if (!LOOP) {
		atlas_smooth_item<TX, TY, ZC>(labels, gnx, gny, tasks, blockTask, blockIdx.x, smooth, crops, ranges);
		return;
	}
	for (unsigned b = blockIdx.x; b < nwork; b += gridDim.x) {
		atlas_smooth_item<TX, TY, ZC>(labels, gnx, gny, tasks, blockTask, b, smooth, crops, ranges);
		__syncthreads(); // the next item reuses the LDS
	}
}

int atlas_tile_count()
{
#define N2M_COUNT_TILE(i, tx, ty, zc) +1
	return 0 N2M_ATLAS_TILES(N2M_COUNT_TILE);
#undef N2M_COUNT_TILE
}

void atlas_tile_shape(int tile, int shape[3])
{
#define N2M_TILE_SHAPE(i, tx, ty, zc)                                                                              \
	if (tile == i) {                                                                                              \
		shape[0] = tx;                                                                                             \
		shape[1] = ty;                                                                                             \
		shape[2] = zc;                                                                                             \
		return;                                                                                                    \
	}
	N2M_ATLAS_TILES(N2M_TILE_SHAPE)
#undef N2M_TILE_SHAPE
	shape[0] = SM_TX;
	shape[1] = SM_TY;
	shape[2] = SM_ZC;
}

void launch_atlas_smooth(const float *labels, int gnx, int gny, int gnz, const AtlasTask *tasks,
                         const uint32_t *blockTask, unsigned nblocks, unsigned grid, int smooth, int tile,
                         float *crops, uint32_t *ranges, hipStream_t s)
{
	if (!nblocks)
		return;
#define N2M_LAUNCH_TILE(i, tx, ty, zc)                                                                             \
	if (tile == i) {                                                                                              \
		if (grid < nblocks)                                                                                        \
			hipLaunchKernelGGL((k_atlas_smooth<tx, ty, zc, true>), dim3(grid), dim3(SM_BS), 0, s, labels, gnx, gny, \
			                   tasks, blockTask, nblocks, smooth, crops, ranges);                                   \
		else                                                                                                       \
			hipLaunchKernelGGL((k_atlas_smooth<tx, ty, zc, false>), dim3(nblocks), dim3(SM_BS), 0, s, labels, gnx,  \
			                   gny, tasks, blockTask, nblocks, smooth, crops, ranges);                              \
		return;                                                                                                    \
	}
	N2M_ATLAS_TILES(N2M_LAUNCH_TILE)
#undef N2M_LAUNCH_TILE
}

// darken the voxels on the volume's faces, bounding box of >= iso and the
// minimum of the result, per task (src/meshify.c:347-371).  Bound by its reads
// once a workgroup takes enough voxels: with 4 per thread, a division for
// each and the workgroups' box atomics four times as many, 370 crops with
// 20.3 M voxels took 198 us, 16 per thread 58.
constexpr int AA_VPT = 16;
__device__ __forceinline__ void atlas_apply_item(float *__restrict__ crops, int gnx, int gny, int gnz,
                                                 const AtlasTask *__restrict__ tasks,
                                                 const uint32_t *__restrict__ blockTask, unsigned b,
                                                 int *__restrict__ bbox, uint32_t *__restrict__ vmin)
{
	__shared__ int s_red[6][4];
	__shared__ uint32_t s_min[4];
	const int ti = (int)blockTask[b];
	const AtlasTask t = tasks[ti];
	const int local = (int)b - t.first_block;
	const size_t n = (size_t)t.nx * t.ny * t.nz;
	float lmin = __builtin_inff();
	int bmin[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, bmax[3] = {-1, -1, -1};
	float *img = crops + t.off;
	// AA_VPT voxels per thread, the workgroup's threads side by side; the
	// coordinates are divided out once and stepped from there
	const size_t v0 = (size_t)local * AA_VPT * 256 + threadIdx.x;
	const int dx = 256 % t.nx, sy = 256 / t.nx, dy = sy % t.ny, dz = sy / t.ny;
	const size_t r0 = v0 / t.nx;
	int x = (int)(v0 - r0 * t.nx), y = (int)(r0 % t.ny), z = (int)(r0 / t.ny);
	for (int k0 = 0; k0 < AA_VPT; k0 += 8) {
		float in[8];
#pragma unroll
		for (int k = 0; k < 8; k++) {
			const size_t v = v0 + (size_t)(k0 + k) * 256;
			in[k] = v < n ? img[v] : 0.f;
		}
#pragma unroll
		for (int k = 0; k < 8; k++) {
			const size_t v = v0 + (size_t)(k0 + k) * 256;
			if (v < n) {
				float val = in[k];
				if (val >= t.iso) {
					bmin[0] = min(bmin[0], x);
					bmax[0] = max(bmax[0], x);
					bmin[1] = min(bmin[1], y);
					bmax[1] = max(bmax[1], y);
					bmin[2] = min(bmin[2], z);
					bmax[2] = max(bmax[2], z);
				}
				const int gx = t.ox + x, gy = t.oy + y, gz = t.oz + z;
				if (gx == 0 || gy == 0 || gz == 0 || gx == gnx - 1 || gy == gny - 1 || gz == gnz - 1) {
					val = fminf(t.edgeMax, val);
					img[v] = val;
				}
				lmin = fminf(lmin, val);
			}
			x += dx;
			y += dy;
			z += dz;
			if (x >= t.nx) {
				x -= t.nx;
				y++;
			}
			if (y >= t.ny) {
				y -= t.ny;
				z++;
			}
		}
	}
	for (int k = 0; k < 3; k++) {
		bmin[k] = wave_min_i32(bmin[k]);
		bmax[k] = wave_max_i32(bmax[k]);
	}
	uint32_t om = wave_min_u32(f2ord(lmin));
	if (lane_id() == 0) {
		for (int k = 0; k < 3; k++) {
			s_red[k][wave_id()] = bmin[k];
			s_red[3 + k][wave_id()] = bmax[k];
		}
		s_min[wave_id()] = om;
	}
	__syncthreads();
	int *bb = bbox + 6 * ti;
	if (threadIdx.x < 6) {
		int k = threadIdx.x;
		int r = s_red[k][0];
		for (int w = 1; w < 4; w++)
			r = k < 3 ? min(r, s_red[k][w]) : max(r, s_red[k][w]);
		const int cur = (int)ld_agent((const uint32_t *)&bb[k]);
		if (k < 3) {
			if (r != 0x7fffffff && r < cur)
				atomicMin(&bb[k], r);
		} else if (r >= 0 && r > cur) {
			atomicMax(&bb[k], r);
		}
	}
	if (threadIdx.x == 6) {
		uint32_t m = min(min(s_min[0], s_min[1]), min(s_min[2], s_min[3]));
		if (m < ld_agent(&vmin[ti]))
			atomicMin(&vmin[ti], m);
	}
}

template <bool LOOP>
__global__ void __launch_bounds__(256)
k_atlas_apply(float *__restrict__ crops, int gnx, int gny, int gnz, const AtlasTask *__restrict__ tasks,
              const uint32_t *__restrict__ blockTask, unsigned nwork, int *__restrict__ bbox,
              uint32_t *__restrict__ vmin)
{
	if (!LOOP) {
		atlas_apply_item(crops, gnx, gny, gnz, tasks, blockTask, blockIdx.x, bbox, vmin);
		return;
	}
	for (unsigned b = blockIdx.x; b < nwork; b += gridDim.x) { // persistent, as k_atlas_smooth
		atlas_apply_item(crops, gnx, gny, gnz, tasks, blockTask, b, bbox, vmin);
		__syncthreads(); // the next item rewrites the LDS partials
	}
}

__global__ void k_atlas_iso(AtlasTask *__restrict__ tasks, int ntasks, const uint32_t *__restrict__ ranges, float req)
{
	const int t = blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= ntasks)
		return;
	const float mn = ord2f(ranges[2 * t]), mx = ord2f(ranges[2 * t + 1]);
	float iso = __builtin_nanf(""), edge = __builtin_nanf("");
	bool fb;
	atlas_iso(req, mn, mx, &iso, &edge, &fb);
	tasks[t].iso = iso;
	tasks[t].mn = mn;
	tasks[t].edgeMax = edge;
}

void launch_atlas_iso(AtlasTask *tasks, int ntasks, const uint32_t *ranges, float req, hipStream_t s)
{
	if (ntasks)
		hipLaunchKernelGGL(k_atlas_iso, dim3((ntasks + 255) / 256), dim3(256), 0, s, tasks, ntasks, ranges, req);
}

void launch_atlas_apply(float *crops, int gnx, int gny, int gnz, const AtlasTask *tasks, const uint32_t *blockTask,
                        unsigned nblocks, unsigned grid, int *bbox, uint32_t *vmin, hipStream_t s)
{
	if (nblocks && grid < nblocks)
		hipLaunchKernelGGL(k_atlas_apply<true>, dim3(grid), dim3(256), 0, s, crops, gnx, gny, gnz, tasks, blockTask,
		                   nblocks, bbox, vmin);
	else if (nblocks)
		hipLaunchKernelGGL(k_atlas_apply<false>, dim3(nblocks), dim3(256), 0, s, crops, gnx, gny, gnz, tasks,
		                   blockTask, nblocks, bbox, vmin);
}

// Planes per workgroup of the smoothing: SM_ZC, halved (down to SM_ZMIN) until
// the launch has SM_WGS workgroups.  A workgroup's planes follow one
// another (about 1.6 us each), so a small volume takes as long as its longest
// chunk; each chunk reads 4 planes more than it writes, so a launch that
// fills the chip keeps the long ones.  128^3: 61 us with 32 planes, 23 with
// 4; 142 x 178 x 142: 69 and 39 (8 planes); 256^3: 92 and 90 (16 planes).
constexpr int SM_ZMIN = 4;
constexpr size_t SM_WGS = 2048;
static int smooth_chunk(size_t columns, int nz)
{
	int zc = SM_ZC;
	while (zc > SM_ZMIN && columns * ((nz + zc - 1) / zc) < SM_WGS)
		zc /= 2;
	return zc;
}

void launch_smooth(const float *in, float *out, int nx, int ny, int nz, uint32_t *range, const float *isos,
                   int nmask, uint32_t *bits, hipStream_t s)
{
	dim3 grid((nx + SM_TX - 1) / SM_TX, (ny + SM_TY - 1) / SM_TY, 1);
	const int zc = smooth_chunk((size_t)grid.x * grid.y, nz);
	grid.z = (nz + zc - 1) / zc;
	int W = (nx + 31) / 32;
	IsoMasks m{};
	m.n = bits ? (nmask < N2M_SMOOTH_MASKS ? nmask : N2M_SMOOTH_MASKS) : 0;
	for (int k = 0; k < m.n; k++)
		m.v[k] = isos[k];
	m.nwords = (size_t)W * ny * nz;
	hipLaunchKernelGGL(k_smooth, grid, dim3(SM_BS), 0, s, in, out, nx, ny, nz, zc, range, m, bits, W);
}

__global__ void k_put(uint32_t *__restrict__ dst, PutWords w, int n)
{
	if ((int)threadIdx.x < n)
		dst[threadIdx.x] = w.v[threadIdx.x];
}

void launch_put(uint32_t *dst, const PutWords &w, int n, hipStream_t s)
{
	hipLaunchKernelGGL(k_put, dim3(1), dim3(64), 0, s, dst, w, n);
}

// ---------------------------------------------------------------------------
// Intensity range without smoothing (src/meshify.c:306-311).
// ---------------------------------------------------------------------------
constexpr int MM_BS = 1024, MM_WGS = 256;
__global__ void __launch_bounds__(MM_BS)
k_minmax(const float *__restrict__ img, size_t n, int vec4, uint32_t *range)
{
	constexpr int NW = MM_BS / N2M_WAVE;
	__shared__ uint32_t s_red[2][NW];
	float lmin = __builtin_inff(), lmax = -__builtin_inff();
	const size_t n4 = vec4 ? n / 4 : 0, tid = blockIdx.x * (size_t)MM_BS + threadIdx.x, step = (size_t)gridDim.x * MM_BS;
	const float4 *v4 = reinterpret_cast<const float4 *>(img);
#pragma unroll 4
	for (size_t i = tid; i < n4; i += step) {
		const float4 v = v4[i];
		lmin = fminf(fminf(lmin, v.x), fminf(v.y, fminf(v.z, v.w)));
		lmax = fmaxf(fmaxf(lmax, v.x), fmaxf(v.y, fmaxf(v.z, v.w)));
	}
	for (size_t i = n4 * 4 + tid; i < n; i += step) {
		lmin = fminf(lmin, img[i]);
		lmax = fmaxf(lmax, img[i]);
	}
	uint32_t omin = wave_min_u32(f2ord(lmin)), omax = wave_max_u32(f2ord(lmax));
	if (lane_id() == 0) {
		s_red[0][wave_id()] = omin;
		s_red[1][wave_id()] = omax;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		for (int w = 1; w < NW; w++) {
			omin = min(omin, s_red[0][w]);
			omax = max(omax, s_red[1][w]);
		}
		// same-address atomics serialise across the chip: only a block that
		// improves on what it reads issues one
		if (omin < ld_agent(&range[0]))
			atomicMin(&range[0], omin);
		if (omax > ld_agent(&range[1]))
			atomicMax(&range[1], omax);
	}
}

// one workgroup of 1024 per CU at most, few atomics (256^3: 29 us with 2048 of
// 256, 20 so)
void launch_minmax(const float *img, size_t n, uint32_t *range, hipStream_t s)
{
	size_t blocks = (n / 4 + MM_BS - 1) / MM_BS;
	blocks = blocks < 1 ? 1 : (blocks > (size_t)MM_WGS ? (size_t)MM_WGS : blocks);
	int vec4 = ((uintptr_t)img & 15) == 0; // float4 loads need 16-byte alignment
	hipLaunchKernelGGL(k_minmax, dim3((unsigned)blocks), dim3(MM_BS), 0, s, img, n, vec4, range);
}

// the block map of a launch over all tasks: task k's workgroups
// [tasks[k].first_block, + count[k]) name it
__global__ void k_atlas_bmap(const AtlasTask *__restrict__ tasks, int ntasks, uint32_t nblocks, uint32_t *__restrict__ bmap)
{
	const int k = blockIdx.x;
	const uint32_t b0 = (uint32_t)tasks[k].first_block,
	               b1 = k + 1 < ntasks ? (uint32_t)tasks[k + 1].first_block : nblocks;
	for (uint32_t b = b0 + threadIdx.x; b < b1; b += blockDim.x)
		bmap[b] = (uint32_t)k;
}

void launch_atlas_bmap(const AtlasTask *tasks, int ntasks, uint32_t nblocks, uint32_t *bmap, hipStream_t s)
{
	if (ntasks)
		hipLaunchKernelGGL(k_atlas_bmap, dim3(ntasks), dim3(256), 0, s, tasks, ntasks, nblocks, bmap);
}

// ---------------------------------------------------------------------------
// Threshold mask bits: bit = (img >= iso) (or img != 0 when `nonzero`), the
// masks of all isolevels of `iso` in one read, mask k to bits + k * iso.nwords.
// range / only_moved: see launch_mask_bits (one isolevel).
// ---------------------------------------------------------------------------
// the isolevel of a mask (launch_mask_bits); false: the mask stays.  Without
// variability no voxel passes: the labelling is queued before the host knows
// the range, and the mask it reads has to have been written.
__device__ __forceinline__ bool mask_iso(const uint32_t *range, int only_moved, float &iso)
{
	if (!range)
		return true;
	float edgeMax;
	bool moved = false;
	if (!atlas_iso(iso, ord2f(range[0]), ord2f(range[1]), &iso, &edgeMax, &moved))
		iso = __builtin_nanf("");
	return moved || !only_moved;
}

// Any row length: a wave takes 64 consecutive voxels of a row (an item; the
// items of a row are ceil(nx / 64)), MB_IN items in flight.  245 x 347 x 275,
// three isolevels: 130 us in three passes of one workgroup per row, 49 so.
constexpr int MB_IN = 4;
__global__ void __launch_bounds__(256)
k_mask_bits(const float *__restrict__ img, int nx, size_t rows, int W, IsoMasks iso, int nonzero,
            uint32_t *__restrict__ bits, const uint32_t *__restrict__ range, int only_moved)
{
	float iso0 = iso.v[0]; // the others stay among the arguments
	if (!mask_iso(range, only_moved, iso0))
		return;
	const int lane = lane_id(), nch = (nx + N2M_WAVE - 1) / N2M_WAVE;
	const size_t items = rows * nch, step = (size_t)gridDim.x * (256 / N2M_WAVE) * MB_IN;
	for (size_t it = ((size_t)blockIdx.x * (256 / N2M_WAVE) + wave_id()) * MB_IN; it < items; it += step) {
		size_t row = it / nch;
		int ch = (int)(it - row * nch);
		float v[MB_IN];
		bool in[MB_IN];
		size_t wi[MB_IN];
		int w1[MB_IN]; // words of the item inside the row
#pragma unroll
		for (int k = 0; k < MB_IN; k++) {
			const int x = ch * N2M_WAVE + lane;
			in[k] = it + k < items && x < nx;
			v[k] = in[k] ? img[row * nx + x] : 0.f;
			wi[k] = row * W + 2 * ch;
			w1[k] = it + k < items ? (2 * ch + 1 < W ? 2 : 1) : 0;
			if (++ch == nch) {
				ch = 0;
				row++;
			}
		}
#pragma unroll
		for (int k = 0; k < MB_IN; k++)
			for (int q = 0; q < iso.n; q++) {
				const unsigned long long m = __ballot(in[k] && (nonzero ? v[k] != 0.0f : v[k] >= (q ? iso.v[q] : iso0)));
				if (lane < w1[k])
					bits[q * iso.nwords + wi[k] + lane] = (uint32_t)(lane ? m >> 32 : m);
			}
	}
}

// The same with 16-byte loads, for rows of a multiple of 32 voxels (nx = 32W)
// whose 16-byte chunks (lpr = nx/4 per row) either fit a workgroup (several
// rows per pass) or fill whole passes of it.  A lane tests 4 voxels; 8
// neighbouring lanes OR their nibbles into a word.
__global__ void __launch_bounds__(256)
k_mask_bits4(const float *__restrict__ img, int nx, size_t rows, int W, IsoMasks iso, int nonzero,
             uint32_t *__restrict__ bits, const uint32_t *__restrict__ range, int only_moved)
{
	float iso0 = iso.v[0]; // the others stay among the arguments
	if (!mask_iso(range, only_moved, iso0))
		return;
	const int lpr = nx >> 2, span = lpr < (int)blockDim.x ? lpr : (int)blockDim.x;
	const int rpi = (int)blockDim.x / span, sub = threadIdx.x / span, q0 = threadIdx.x % span;
	for (size_t row0 = (size_t)blockIdx.x * rpi; row0 < rows; row0 += (size_t)gridDim.x * rpi) {
		const size_t row = row0 + sub;
		const bool live = sub < rpi && row < rows;
		for (int q = q0; q < lpr; q += span) { // the same trip count on every lane
			float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
			if (live)
				v = reinterpret_cast<const float4 *>(img + row * nx)[q];
			for (int k = 0; k < iso.n; k++) {
				const float t = k ? iso.v[k] : iso0;
				uint32_t nib = 0;
				if (live && nonzero)
					nib = (v.x != 0.0f) | (v.y != 0.0f) << 1 | (v.z != 0.0f) << 2 | (v.w != 0.0f) << 3;
				else if (live)
					nib = (v.x >= t) | (v.y >= t) << 1 | (v.z >= t) << 2 | (v.w >= t) << 3;
				uint32_t wv = nib << (4 * (q & 7));
				wv |= __shfl_xor(wv, 1, N2M_WAVE);
				wv |= __shfl_xor(wv, 2, N2M_WAVE);
				wv |= __shfl_xor(wv, 4, N2M_WAVE);
				if (live && (q & 7) == 0)
					bits[k * iso.nwords + (size_t)W * row + (q >> 3)] = wv;
			}
		}
	}
}

static unsigned row_blocks(size_t rows) { return (unsigned)(rows < 8192 ? (rows ? rows : 1) : 8192); }

static void mask_pass(const float *img, int nx, int ny, int nz, const IsoMasks &m, int nonzero, uint32_t *bits,
                      const uint32_t *range, int only_moved, hipStream_t s)
{
	const int W = (nx + 31) / 32, lpr = nx / 4;
	const size_t rows = (size_t)ny * nz;
	// a pass that nearly always has nothing to do is launched small
	const unsigned most = only_moved ? 512 : 4096;
	if (nx % 32 == 0 && (reinterpret_cast<uintptr_t>(img) & 15u) == 0 && (lpr <= 256 || lpr % 256 == 0)) {
		const size_t rpi = lpr < 256 ? 256 / lpr : 1;
		const unsigned nb = row_blocks((rows + rpi - 1) / rpi);
		hipLaunchKernelGGL(k_mask_bits4, dim3(only_moved && nb > most ? most : nb), dim3(256), 0, s, img, nx, rows, W, m,
		                   nonzero, bits, range, only_moved);
	} else {
		const size_t items = rows * ((nx + N2M_WAVE - 1) / N2M_WAVE), per = 256 / N2M_WAVE * MB_IN;
		const size_t nb = (items + per - 1) / per;
		hipLaunchKernelGGL(k_mask_bits, dim3((unsigned)(nb < most ? (nb ? nb : 1) : most)), dim3(256), 0, s, img, nx,
		                   rows, W, m, nonzero, bits, range, only_moved);
	}
}

void launch_mask_bits_multi(const float *img, int nx, int ny, int nz, const float *isos, int n, uint32_t *bits,
                            hipStream_t s)
{
	IsoMasks m{};
	m.nwords = (size_t)((nx + 31) / 32) * ny * nz;
	for (int k0 = 0; k0 < n; k0 += N2M_SMOOTH_MASKS) {
		m.n = n - k0 < N2M_SMOOTH_MASKS ? n - k0 : N2M_SMOOTH_MASKS;
		for (int k = 0; k < m.n; k++)
			m.v[k] = isos[k0 + k];
		mask_pass(img, nx, ny, nz, m, 0, bits + k0 * m.nwords, nullptr, 0, s);
	}
}

void launch_mask_bits(const float *img, int nx, int ny, int nz, float iso, int nonzero, uint32_t *bits,
                      hipStream_t s, const uint32_t *range, bool only_moved)
{
	IsoMasks m{};
	m.n = 1;
	m.v[0] = iso;
	mask_pass(img, nx, ny, nz, m, nonzero, bits, range, only_moved ? 1 : 0, s);
}

// ---------------------------------------------------------------------------
// dilate(mask, dim, true), src/meshify.c:218-264: a voxel at least one away
// from every face is switched on if any of its 26 neighbours except
// (-1,-1,-1) is on.  One thread per word.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t word_at(const uint32_t *bits, int W, int ny, int wx, int y, int z)
{
	return (wx >= 0 && wx < W) ? bits[(size_t)wx + (size_t)W * ((size_t)y + (size_t)ny * z)] : 0u;
}

__global__ void __launch_bounds__(256)
k_dilate_bits(const uint32_t *__restrict__ in, uint32_t *__restrict__ out, int nx, int ny, int nz, int W)
{
	size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
	size_t nw = (size_t)W * ny * nz;
	if (t >= nw)
		return;
	const int wx = (int)(t % W);
	const size_t row = t / W;
	const int y = (int)(row % ny), z = (int)(row / ny);
	uint32_t self = in[t];
	uint32_t acc = 0;
	if (y >= 1 && y < ny - 1 && z >= 1 && z < nz - 1) {
		for (int dz = -1; dz <= 1; dz++)
			for (int dy = -1; dy <= 1; dy++) {
				uint32_t c = word_at(in, W, ny, wx, y + dy, z + dz);
				uint32_t p = word_at(in, W, ny, wx - 1, y + dy, z + dz);
				uint32_t n = word_at(in, W, ny, wx + 1, y + dy, z + dz);
				uint32_t xm = (c << 1) | (p >> 31); // neighbour at x-1
				uint32_t xp = (c >> 1) | (n << 31); // neighbour at x+1
				if (dz == -1 && dy == -1)
					acc |= c | xp; // (-1,-1,-1) is not tested
				else if (dz == 0 && dy == 0)
					acc |= xm | xp;
				else
					acc |= xm | c | xp;
			}
		// interior in x: 1 <= x <= nx-2
		uint32_t xmask = 0xffffffffu;
		int xb = wx * 32;
		for (int b = 0; b < 32; b++) {
			int xx = xb + b;
			if (xx < 1 || xx > nx - 2)
				xmask &= ~(1u << b);
		}
		acc &= xmask;
	}
	out[t] = self | acc;
}

void launch_dilate_bits(const uint32_t *in, uint32_t *out, int nx, int ny, int nz, hipStream_t s)
{
	int W = (nx + 31) / 32;
	size_t nw = (size_t)W * ny * nz;
	hipLaunchKernelGGL(k_dilate_bits, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, s, in, out, nx, ny,
	                   nz, W);
}

// ---------------------------------------------------------------------------
// Apply (src/meshify.c:332-371): raise filled voxels to iso, set voxels
// outside the dilated largest cluster to mn, record the bounding box of
// voxels >= iso, then clamp the outer faces to edgeMax.
// keep: mask after bwlabel (fill target); dil: dilated mask (or null).
// The box is {minx,miny,minz,maxx,maxy,maxz}.
// ---------------------------------------------------------------------------
// Box and minimum are reduced through one row of partial results per
// workgroup and a one-workgroup launch, which hands them to the host by
// itself: with atomics on one line from every workgroup this pass took
// 40 us on a 128^3 volume (8 MiB) and 97 on a 256^3 one; now 7 and 37, and
// 5.6 for the small launch, which takes the place of a copy.
constexpr int AP_WORDS = 7, AP_MAXWG = 1024;

// Division of 32-bit numbers by a fixed one (multiply and shift; the method of
// Granlund and Montgomery, "Division by invariant integers using
// multiplication", 1994)
struct FixedDiv {
	uint32_t m, s1, s2;
	explicit FixedDiv(uint32_t d)
	{
		uint32_t l = 0;
		while (l < 32 && (1ull << l) < d)
			l++;
		m = (uint32_t)(((1ull << 32) * ((1ull << l) - d)) / d + 1);
		s1 = l < 1 ? l : 1;
		s2 = l > 1 ? l - 1 : 0;
	}
	__device__ uint32_t operator()(uint32_t n) const
	{
		const uint32_t t = __umulhi(m, n);
		return (t + ((n - t) >> s1)) >> s2;
	}
};

// What the apply stage does to one voxel, and the box and minimum it keeps.
// kw / dw: the keep / dilated-mask words that hold bit x & 31.
struct ApplyVoxel {
	float iso, mn, edgeMax;
	int nx;
	bool k_on, d_on;
	float lmin = __builtin_inff();
	int bmin[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, bmax[3] = {-1, -1, -1};

	__device__ __forceinline__ float operator()(int x, int y, int z, bool face_row, float val, uint32_t kw, uint32_t dw)
	{
		if (k_on && ((kw >> (x & 31)) & 1u))
			val = (float)fmax((double)val, (double)iso);
		if (d_on && !((dw >> (x & 31)) & 1u))
			val = mn;
		if (val >= iso) {
			bmin[0] = min(bmin[0], x);
			bmax[0] = max(bmax[0], x);
			bmin[1] = min(bmin[1], y);
			bmax[1] = max(bmax[1], y);
			bmin[2] = min(bmin[2], z);
			bmax[2] = max(bmax[2], z);
		}
		if (face_row || x == 0 || x == nx - 1)
			val = fminf(edgeMax, val);
		lmin = fminf(lmin, val);
		return val;
	}

	// the workgroup's box and minimum to its column of part
	__device__ __forceinline__ void store(uint32_t *__restrict__ part)
	{
		__shared__ int s_red[6][4];
		__shared__ uint32_t s_min[4];
		for (int k = 0; k < 3; k++) {
			bmin[k] = wave_min_i32(bmin[k]);
			bmax[k] = wave_max_i32(bmax[k]);
		}
		const uint32_t om = wave_min_u32(f2ord(lmin));
		if (lane_id() == 0) {
			for (int k = 0; k < 3; k++) {
				s_red[k][wave_id()] = bmin[k];
				s_red[3 + k][wave_id()] = bmax[k];
			}
			s_min[wave_id()] = om;
		}
		__syncthreads();
		if (threadIdx.x < 6) {
			const int k = threadIdx.x;
			int r = s_red[k][0];
			for (int w = 1; w < 4; w++)
				r = k < 3 ? min(r, s_red[k][w]) : max(r, s_red[k][w]);
			part[k * AP_MAXWG + blockIdx.x] = (uint32_t)r;
		}
		if (threadIdx.x == 6)
			part[6 * AP_MAXWG + blockIdx.x] = min(min(s_min[0], s_min[1]), min(s_min[2], s_min[3]));
	}
};

// the sign bits of 4 voxels of the Lewiner data lw_clamp(v - iso), whose 8
// lanes (lane & 7 = part) together hold a word; lane 0 of them writes it
__device__ __forceinline__ void apply_signs(const float (&vv)[4], int nlive, float iso, int part, size_t word,
                                            uint32_t *__restrict__ sgp, uint32_t *__restrict__ sgn)
{
	uint32_t bp = 0, bn = 0;
#pragma unroll
	for (int u = 0; u < 4; u++) {
		float d = vv[u] - iso;
		d = fabsf(d) < FLT_EPSILON ? FLT_EPSILON : d;
		bp |= (uint32_t)(u < nlive && d > 0.f) << u;
		bn |= (uint32_t)(u < nlive && d < 0.f) << u;
	}
	bp <<= 4 * part;
	bn <<= 4 * part;
#pragma unroll
	for (int m = 1; m < 8; m <<= 1) {
		bp |= __shfl_xor(bp, m);
		bn |= __shfl_xor(bn, m);
	}
	if (part == 0) {
		sgp[word] = bp;
		sgn[word] = bn;
	}
}

// row by row; vec4: 16-byte loads and stores (rows of nx = 4 * lpr voxels).
// sgp / sgn (vec4, nx % 32 == 0): the sign bits.
__global__ void __launch_bounds__(256)
k_apply(const float *src, float *img, int nx, int ny, int nz, int W, int vec4, float iso, float mn,
        float edgeMax, const uint32_t *__restrict__ keep, const uint32_t *__restrict__ dil, int fill,
        const uint32_t *__restrict__ range, uint32_t *__restrict__ part, uint32_t *__restrict__ sgp,
        uint32_t *__restrict__ sgn)
{
	if (range) {
		bool moved;
		mn = ord2f(range[0]);
		if (!atlas_iso(iso, mn, ord2f(range[1]), &iso, &edgeMax, &moved))
			return;
	}
	const size_t rows = (size_t)ny * nz;
	const bool k_on = fill && keep, d_on = dil != nullptr;
	ApplyVoxel voxel{iso, mn, edgeMax, nx, k_on, d_on};
	if (vec4) {
		// several rows per pass when a row has fewer 16-byte chunks than the
		// workgroup has threads
		const int lpr = nx >> 2, span = lpr < (int)blockDim.x ? lpr : (int)blockDim.x;
		const int rpi = (int)blockDim.x / span, sub = threadIdx.x / span, q0 = threadIdx.x % span;
		for (size_t row0 = (size_t)blockIdx.x * rpi; row0 < rows; row0 += (size_t)gridDim.x * rpi) {
			const size_t row = row0 + sub;
			if (sub >= rpi || row >= rows)
				continue;
			const int y = (int)(row % ny), z = (int)(row / ny);
			const bool face_row = y == 0 || z == 0 || y == ny - 1 || z == nz - 1;
			const float4 *in = reinterpret_cast<const float4 *>(src + row * nx);
			float4 *line = reinterpret_cast<float4 *>(img + row * nx);
			for (int q = q0; q < lpr; q += span) {
				const int x = 4 * q;
				const uint32_t kw = k_on ? keep[(size_t)W * row + (x >> 5)] : 0u;
				const uint32_t dw = d_on ? dil[(size_t)W * row + (x >> 5)] : 0u;
				const float4 v = in[q];
				float vv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
				for (int u = 0; u < 4; u++)
					vv[u] = voxel(x + u, y, z, face_row, vv[u], kw, dw);
				line[q] = make_float4(vv[0], vv[1], vv[2], vv[3]);
				// the 8 lanes of an aligned group hold one 32-voxel word of the
				// row (nx % 32 == 0 and the span a multiple of 8, so the group
				// shares its row and its trip count)
				if (sgp)
					apply_signs(vv, 4, iso, q & 7, (size_t)W * row + (x >> 5), sgp, sgn);
			}
		}
	} else {
		// whole rows per workgroup: y and z are uniform, no per-voxel division
		for (size_t row = blockIdx.x; row < rows; row += gridDim.x) {
			const int y = (int)(row % ny), z = (int)(row / ny);
			const bool face_row = y == 0 || z == 0 || y == ny - 1 || z == nz - 1;
			const float *in = src + row * nx;
			float *line = img + row * nx;
			for (int x = threadIdx.x; x < nx; x += blockDim.x) {
				const uint32_t kw = k_on ? keep[(size_t)W * row + (x >> 5)] : 0u;
				const uint32_t dw = d_on ? dil[(size_t)W * row + (x >> 5)] : 0u;
				line[x] = voxel(x, y, z, face_row, in[x], kw, dw);
			}
		}
	}
	voxel.store(part);
}

// The same in linear voxel order, for rows of any length: 16-byte loads and
// stores, 4 voxels per thread wherever its rows begin, so that the sign bits
// come out as the classify pass reads them (bit j of the arrays <-> voxel j)
// and rows of odd length need no other classify.  142 x 178 x 142: apply 24 ->
// 15 us, classify (from the values before) 35 -> 20.
__global__ void __launch_bounds__(256)
k_apply_linear(const float *src, float *img, int nx, int ny, int nz, uint32_t nvox, FixedDiv by_nx, FixedDiv by_ny, int W,
               float iso, float mn, float edgeMax, const uint32_t *__restrict__ keep,
               const uint32_t *__restrict__ dil, int fill, const uint32_t *__restrict__ range,
               uint32_t *__restrict__ part, uint32_t *__restrict__ sgp, uint32_t *__restrict__ sgn)
{
	if (range) {
		bool moved;
		mn = ord2f(range[0]);
		if (!atlas_iso(iso, mn, ord2f(range[1]), &iso, &edgeMax, &moved))
			return;
	}
	const bool k_on = fill && keep, d_on = dil != nullptr;
	ApplyVoxel voxel{iso, mn, edgeMax, nx, k_on, d_on};
	const uint32_t nq = (uint32_t)(((unsigned long long)nvox + 31) / 32 * 8); // whole groups of 8 lanes
	for (uint32_t q = blockIdx.x * 256 + threadIdx.x; q < nq; q += gridDim.x * 256) {
		const uint32_t v0 = 4 * q;
		const int nlive = v0 >= nvox ? 0 : (nvox - v0 < 4 ? (int)(nvox - v0) : 4);
		float vv[4] = {0.f, 0.f, 0.f, 0.f};
		if (nlive == 4) {
			const float4 f = reinterpret_cast<const float4 *>(src)[q];
			vv[0] = f.x;
			vv[1] = f.y;
			vv[2] = f.z;
			vv[3] = f.w;
		} else {
			for (int u = 0; u < nlive; u++)
				vv[u] = src[v0 + u];
		}
		uint32_t row = by_nx(v0);
		int x = (int)(v0 - row * (uint32_t)nx), z = (int)by_ny(row), y = (int)(row - (uint32_t)z * (uint32_t)ny);
		uint32_t kw = 0, dw = 0;
#pragma unroll
		for (int u = 0; u < 4; u++) {
			if (u < nlive) {
				if (u == 0 || (x & 31) == 0) {
					kw = k_on ? keep[(size_t)W * row + (x >> 5)] : 0u;
					dw = d_on ? dil[(size_t)W * row + (x >> 5)] : 0u;
				}
				vv[u] = voxel(x, y, z, y == 0 || z == 0 || y == ny - 1 || z == nz - 1, vv[u], kw, dw);
				if (++x == nx) {
					x = 0;
					row++;
					if (++y == ny) {
						y = 0;
						z++;
					}
				}
			}
		}
		if (nlive == 4)
			reinterpret_cast<float4 *>(img)[q] = make_float4(vv[0], vv[1], vv[2], vv[3]);
		else
			for (int u = 0; u < nlive; u++)
				img[v0 + u] = vv[u];
		if (sgp)
			apply_signs(vv, nlive, iso, q & 7, q >> 3, sgp, sgn);
	}
	voxel.store(part);
}

// the workgroups' partial boxes and minima to host[0..6], the range to
// host[7..8]; a box without voxels keeps the reference's start values
// (src/meshify.c:349-351)
__global__ void __launch_bounds__(AP_MAXWG)
k_apply_box(const uint32_t *__restrict__ part, int nwg, int nx, int ny, int nz, const uint32_t *__restrict__ range,
            uint32_t *__restrict__ host)
{
	__shared__ uint32_t s[AP_WORDS][AP_MAXWG / N2M_WAVE];
	const bool in = (int)threadIdx.x < nwg; // (left over from another call when k_apply found no variability)
	const int dim[3] = {nx, ny, nz};
#pragma unroll
	for (int k = 0; k < AP_WORDS; k++) {
		const uint32_t v = in ? part[k * AP_MAXWG + threadIdx.x] : (k < 3 ? 0x7fffffffu : 0xffffffffu);
		const uint32_t r = k < 3 ? (uint32_t)wave_min_i32((int)v) : (k < 6 ? (uint32_t)wave_max_i32((int)v)
		                                                                  : wave_min_u32(v));
		if (lane_id() == 0)
			s[k][wave_id()] = r;
	}
	__syncthreads();
	const int k = threadIdx.x;
	if (k < AP_WORDS) {
		uint32_t r = s[k][0];
		for (int w = 1; w < AP_MAXWG / N2M_WAVE; w++)
			r = k < 3 ? (uint32_t)min((int)r, (int)s[k][w])
			          : (k < 6 ? (uint32_t)max((int)r, (int)s[k][w]) : min(r, s[k][w]));
		if (k < 3)
			r = (uint32_t)min((int)r, dim[k]);
		else if (k < 6)
			r = (uint32_t)max((int)r, 0);
		host[k] = r;
	} else if (k < AP_WORDS + 2 && range) {
		host[k] = range[k - AP_WORDS];
	}
}

size_t apply_part_words() { return (size_t)AP_WORDS * AP_MAXWG; }

bool launch_apply(const float *src, float *img, int nx, int ny, int nz, float iso, float mn, float edgeMax,
                  const uint32_t *keep, const uint32_t *dil, int fill, const uint32_t *range, uint32_t *part,
                  uint32_t *host, hipStream_t s, uint32_t *sgp, uint32_t *sgn)
{
	const int W = (nx + 31) / 32;
	const float *in = src ? src : img;
	const size_t rows = (size_t)ny * nz, nvox = rows * nx;
	const bool aligned = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(img)) & 15u) == 0;
	// by rows where that gives whole words and vectors (or no sign bits are
	// asked for), in linear order otherwise, by single voxels where the
	// volumes are not aligned or have 2^32 voxels
	const bool vec4 = aligned && nx % 4 == 0 && (!sgp || nx % 32 == 0);
	const bool linear = aligned && !vec4 && nvox < 0xffffffe0ull;
	if (!vec4 && !linear)
		sgp = sgn = nullptr;
	const size_t rpi = vec4 && nx / 4 < 256 ? 256 / (nx / 4) : 1;
	const size_t items = linear ? (nvox + 1023) / 1024 : (rows + rpi - 1) / rpi;
	const unsigned nwg = (unsigned)(items < (size_t)AP_MAXWG ? (items ? items : 1) : (size_t)AP_MAXWG);
	if (linear)
		hipLaunchKernelGGL(k_apply_linear, dim3(nwg), dim3(256), 0, s, in, img, nx, ny, nz, (uint32_t)nvox,
		                   FixedDiv((uint32_t)nx), FixedDiv((uint32_t)ny), W, iso, mn, edgeMax, keep, dil, fill, range,
		                   part, sgp, sgn);
	else
		hipLaunchKernelGGL(k_apply, dim3(nwg), dim3(256), 0, s, in, img, nx, ny, nz, W, vec4 ? 1 : 0, iso, mn, edgeMax,
		                   keep, dil, fill, range, part, sgp, sgn);
	hipLaunchKernelGGL(k_apply_box, dim3(1), dim3(AP_MAXWG), 0, s, (const uint32_t *)part, (int)nwg, nx, ny, nz,
	                   range, host);
	return sgp != nullptr;
}

// ---------------------------------------------------------------------------
// Histograms for setThreshold() (src/isolevel.c).
// stats: [0]=ord min, [1]=ord max over non-NaN, [2]=NaN count.
// ---------------------------------------------------------------------------
// f(v) for every voxel of img[0, n), grid-stride; 16-byte loads when img is
// 16-byte aligned (the visiting order does not matter to the callers: min,
// max and counts)
template <typename F> __device__ __forceinline__ void each_voxel(const float *__restrict__ img, size_t n, F f)
{
	const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
	size_t done = 0;
	if ((reinterpret_cast<uintptr_t>(img) & 15u) == 0) {
		const float4 *v4 = reinterpret_cast<const float4 *>(img);
		const size_t n4 = n / 4;
#pragma unroll 2
		for (size_t i = tid; i < n4; i += stride) {
			const float4 q = v4[i];
			f(q.x);
			f(q.y);
			f(q.z);
			f(q.w);
		}
		done = 4 * n4;
	}
	for (size_t i = done + tid; i < n; i += stride)
		f(img[i]);
}

// The range and histogram passes run in at most TH_ROWS workgroups of 1024
// threads, each leaving one row of results that the next launch (one
// workgroup) sums: thousands of workgroups adding to the same range words
// and bins spent most of these passes in atomics (7.1 M voxels, 28 MB: range
// 50 us, each histogram 43; now 11 and 16).
constexpr int TH_BS = 1024, TH_ROWS = 256, TH_BINS = 1001;

static unsigned thr_rows(size_t n)
{
	const size_t b = (n + 65535) / 65536; // below that the rows to sum weigh more
	return (unsigned)(b < 1 ? 1 : (b > (size_t)TH_ROWS ? (size_t)TH_ROWS : b));
}

// rows[3 * workgroup]: ordered min, ordered max over non-NaN, NaN count
__global__ void __launch_bounds__(TH_BS) k_hist_range(const float *__restrict__ img, size_t n, uint32_t *rows)
{
	__shared__ uint32_t s_red[3][TH_BS / N2M_WAVE];
	float lmin = __builtin_inff(), lmax = -__builtin_inff();
	uint32_t nan = 0;
	each_voxel(img, n, [&](float v) {
		if (v != v) {
			nan++;
			return;
		}
		lmin = fminf(lmin, v);
		lmax = fmaxf(lmax, v);
	});
	uint32_t omin = wave_min_u32(f2ord(lmin)), omax = wave_max_u32(f2ord(lmax));
	nan = wave_sum(nan);
	if (lane_id() == 0) {
		s_red[0][wave_id()] = omin;
		s_red[1][wave_id()] = omax;
		s_red[2][wave_id()] = nan;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		for (int w = 1; w < TH_BS / N2M_WAVE; w++) {
			omin = min(omin, s_red[0][w]);
			omax = max(omax, s_red[1][w]);
			nan += s_red[2][w];
		}
		rows[3 * blockIdx.x] = omin;
		rows[3 * blockIdx.x + 1] = omax;
		rows[3 * blockIdx.x + 2] = nan;
	}
}

// rows[nbins * workgroup + bin]; bin = round((v - mn) * scl) in float, clamped
// to [0, nbins-1] (the 1001-bin pass never leaves that range for finite
// data), with mn = par[0], scl = par[1]; nothing when *enable is 0.
__global__ void __launch_bounds__(TH_BS)
k_hist_bins(const float *__restrict__ img, size_t n, const float *__restrict__ par,
            const int32_t *__restrict__ enable, int nbins, uint32_t *__restrict__ rows)
{
	__shared__ uint32_t s_h[TH_BINS];
	if (enable && *enable == 0)
		return;
	const float mn = par[0], scl = par[1];
	for (int i = threadIdx.x; i < nbins; i += TH_BS)
		s_h[i] = 0;
	__syncthreads();
	// bin 0 (most of a background) is counted in a register, a run of voxels in
	// another bin is added with one LDS atomic
	int cb = 0;
	uint32_t cc = 0, c0 = 0;
	each_voxel(img, n, [&](float v) {
		if (v != v)
			return;
		float f = (v - mn) * scl;
		int b = (int)roundf(f);
		b = b < 0 ? 0 : (b > nbins - 1 ? nbins - 1 : b);
		if (b == 0) {
			c0++;
			return;
		}
		if (b == cb) {
			cc++;
			return;
		}
		if (cc)
			atomicAdd(&s_h[cb], cc);
		cb = b;
		cc = 1;
	});
	if (cc)
		atomicAdd(&s_h[cb], cc);
	c0 = wave_sum(c0);
	if (lane_id() == 0 && c0)
		atomicAdd(&s_h[0], c0);
	__syncthreads();
	for (int i = threadIdx.x; i < nbins; i += TH_BS)
		rows[(size_t)nbins * blockIdx.x + i] = s_h[i];
}

unsigned atlas_smooth_blocks(int nx, int ny, int nz, int smooth, int tile)
{
	if (smooth) {
		int sh[3];
		atlas_tile_shape(tile, sh);
		return (unsigned)(((nx + sh[0] - 1) / sh[0]) * ((ny + sh[1] - 1) / sh[1]) * ((nz + sh[2] - 1) / sh[2]));
	}
	return (unsigned)(((size_t)nx * ny * nz + SM_BS - 1) / SM_BS);
}
unsigned atlas_apply_blocks(int nx, int ny, int nz)
{
	return (unsigned)(((size_t)nx * ny * nz + 256 * AA_VPT - 1) / (256 * AA_VPT));
}

// one label of the per-label loop: out = (lo < v < hi), count of ones
// (src/nii2mesh.c:553-563)
__global__ void __launch_bounds__(256)
k_binarize(const float *__restrict__ labels, size_t n, float lo, float hi, float *__restrict__ out,
           uint32_t *__restrict__ count)
{
	uint32_t c = 0;
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
		float v = labels[i];
		bool in = v > lo && v < hi;
		out[i] = in ? 1.0f : 0.0f;
		c += in;
	}
	__shared__ uint32_t s_c[4];
	c = wave_sum(c);
	if (lane_id() == 0)
		s_c[wave_id()] = c;
	__syncthreads();
	if (threadIdx.x == 0) {
		c = s_c[0] + s_c[1] + s_c[2] + s_c[3];
		if (c)
			atomicAdd(count, c);
	}
}

void launch_binarize(const float *labels, size_t n, float lo, float hi, float *out, uint32_t *count, hipStream_t s)
{
	size_t b = (n + 255) / 256;
	b = b > 4096 ? 4096 : (b < 1 ? 1 : b);
	hipLaunchKernelGGL(k_binarize, dim3((unsigned)b), dim3(256), 0, s, labels, n, lo, hi, out, count);
}

// ---------------------------------------------------------------------------
// Three-threshold Otsu search of nii_otsu() mode 5 (src/isolevel.c:176-197)
// over the Liao table, P[u][v] at P[u * su + v * sv].  Workgroup l scans every
// (m, h) for that l; each lane keeps the first strict maximum in h order, the
// workgroup the first in m order, and the host the first in l order -- the
// reference's first occurrence of the maximum in (l, m, h) order.
// The lanes of a wave read consecutive m for one h, so the device chain
// keeps the table column by column (su = 1): row by row every lane reads a
// line of its own.  OT_Q threads share an m, each with every OT_Q-th run of h.
// 81 us -> 14.
// ---------------------------------------------------------------------------
constexpr int OT_Q = 4, OT_RUN = 8;
__global__ void __launch_bounds__(256 * OT_Q)
k_otsu3(const double *__restrict__ P, int su, int sv, int nBin, double *__restrict__ bv, int *__restrict__ bm,
        int *__restrict__ bh)
{
	constexpr int NW = 256 * OT_Q / N2M_WAVE;
	__shared__ double s_col[256 + OT_Q * OT_RUN], s_v[NW];
	__shared__ int s_m[NW], s_h[NW];
	const int tm = threadIdx.x & 255, q = threadIdx.x >> 8;
	const int l = blockIdx.x, m = l + 1 + tm;
	if (threadIdx.x < 256 + OT_Q * OT_RUN)
		s_col[threadIdx.x] =
		    (int)threadIdx.x < nBin - 1 ? P[(size_t)(threadIdx.x + 1) * su + (size_t)255 * sv] : 0.0;
	__syncthreads();
	double best = 0.0;
	int bestH = -1, bestM = m;
	const bool live = m < nBin - 2;
	const double a = live ? P[(size_t)l * sv] + P[(size_t)(l + 1) * su + (size_t)m * sv] : 0.0;
	const double *row = P + (size_t)(live ? m + 1 : 0) * su;
	for (int h0 = m - lane_id() + 1 + q * OT_RUN; h0 < nBin - 1; h0 += OT_Q * OT_RUN) { // from the wave's first m
		double t[OT_RUN];
#pragma unroll
		for (int k = 0; k < OT_RUN; k++)
			t[k] = h0 + k < nBin ? row[(size_t)(h0 + k) * sv] : 0.0;
#pragma unroll
		for (int k = 0; k < OT_RUN; k++) {
			const int h = h0 + k;
			const double v = a + t[k] + s_col[h];
			if (live && h > m && h < nBin - 1 && (bestH < 0 || v > best)) {
				best = v;
				bestH = h;
			}
		}
	}
	// the first maximum in (m, h) order: larger value, then smaller m, then h
	auto take = [&](double v, int vm, int vh) {
		if (vh >= 0 && (bestH < 0 || v > best || (v == best && (vm < bestM || (vm == bestM && vh < bestH))))) {
			best = v;
			bestM = vm;
			bestH = vh;
		}
	};
#pragma unroll
	for (int d = N2M_WAVE / 2; d > 0; d >>= 1) {
		const double v = __shfl_xor(best, d);
		const int vm = __shfl_xor(bestM, d), vh = __shfl_xor(bestH, d);
		take(v, vm, vh);
	}
	if (lane_id() == 0) {
		s_v[wave_id()] = best;
		s_m[wave_id()] = bestM;
		s_h[wave_id()] = bestH;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		for (int w = 1; w < NW; w++)
			take(s_v[w], s_m[w], s_h[w]);
		bv[l] = bestH < 0 ? 0.0 : best;
		bm[l] = bestH < 0 ? -1 : bestM;
		bh[l] = bestH;
	}
}

void launch_otsu3(const double *P, int nBin, double *bv, int *bm, int *bh, hipStream_t s)
{
	if (nBin > 3)
		hipLaunchKernelGGL(k_otsu3, dim3(nBin - 3), dim3(256 * OT_Q), 0, s, P, nBin, 1, nBin, bv, bm, bh);
}

// The 256-bin histogram summed from its rows, and the running sums of
// nii_otsu's Liao table (src/isolevel.c:147-165) in the reference's order: the
// bin probabilities in parallel, the sums by one thread (P[0] is the raw
// count H[0], a quirk the thresholds depend on); sums[0..255] = P,
// sums[256..511] = S.
__global__ void __launch_bounds__(TH_BS)
k_otsu_sums(const uint32_t *__restrict__ rows, int nrows, uint32_t *__restrict__ H, double *__restrict__ sums)
{
	constexpr int n = 256;
	__shared__ uint32_t s_part[TH_BS];
	__shared__ double s_prob[n], s_w[n], s_red[n / N2M_WAVE];
	const int v = threadIdx.x % n, q = threadIdx.x / n; // four threads per bin
	uint32_t c = 0;
#pragma unroll 32
	for (int r = q; r < nrows; r += TH_BS / n)
		c += rows[(size_t)n * r + v];
	s_part[threadIdx.x] = c;
	__syncthreads();
	double h = 0.0;
	if (threadIdx.x < n) {
		c = s_part[v] + s_part[n + v] + s_part[2 * n + v] + s_part[3 * n + v];
		H[v] = c;
		h = (double)(int)c;
		const double t = wave_sum(h); // whole numbers: exact in any order
		if (lane_id() == 0)
			s_red[wave_id()] = t;
	}
	__syncthreads();
	if (threadIdx.x < n) {
		const double Sum = s_red[0] + s_red[1] + s_red[2] + s_red[3];
		const double prob = h / Sum;
		s_prob[v] = v ? prob : h;
		s_w[v] = v ? (v + 1) * prob : h;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		double p = s_prob[0], w = s_w[0];
		sums[0] = p;
		sums[n] = w;
#pragma unroll 16
		for (int i = 1; i < n; i++) {
			p = p + s_prob[i];
			w = w + s_w[i];
			sums[i] = p;
			sums[n + i] = w;
		}
	}
}

// The Liao table (src/isolevel.c:166-175), column by column: entry (u, v) at
// PT[v * 256 + u] = (S*S)/P of the bin range [u, v] (left as is when P is 0);
// entries with v < u are never read and are set to 0.  probe: the entries the
// host-side searches read: row 0, column 255 shifted by one row and the four
// terms of the mode-5 start value (lo, mi, hi = 64, 128, 192).
__global__ void __launch_bounds__(256)
k_otsu_table(const double *__restrict__ sums, double *__restrict__ PT, double *__restrict__ probe)
{
	constexpr int n = 256;
	const int v = blockIdx.x, u = threadIdx.x;
	double val = 0.0;
	if (v >= u) {
		const double p = u == 0 ? sums[v] : sums[v] - sums[u - 1];
		const double q = u == 0 ? sums[n + v] : sums[n + v] - sums[n + u - 1];
		val = p != 0 ? (q * q) / p : p;
	}
	PT[(size_t)v * n + u] = val;
	if (u == 0)
		probe[v] = val;
	if (v == n - 1) {
		if (u > 0)
			probe[n + u - 1] = val;
		else
			probe[2 * n - 1] = 0.0;
	}
	if (u == 0 && v == 64)
		probe[2 * n] = val;
	else if (u == 65 && v == 128)
		probe[2 * n + 1] = val;
	else if (u == 129 && v == 192)
		probe[2 * n + 2] = val;
	else if (u == 193 && v == 255)
		probe[2 * n + 3] = val;
}

// ---------------------------------------------------------------------------
// setThreshold() as one chain of launches (src/isolevel.c:35-277), results
// in a ThrRecord.
// ---------------------------------------------------------------------------
// The cases of the robust range (src/isolevel.c:59-139).  First launch
// (final = 0): the range from its rows, and whether the 1001-bin pass runs,
// with its mn and scl.  Second launch: the percentiles (the walk over that
// histogram, summed from its rows, when it ran) and the 256-bin pass's mn and
// scl (src/isolevel.c:245-250).  All float and double arithmetic in the host
// code's order.
__global__ void __launch_bounds__(TH_BS)
k_thr_range(ThrRecord *__restrict__ r, const uint32_t *__restrict__ rows, int nrows, size_t nvox, int final)
{
	constexpr int kBins = TH_BINS;
	__shared__ uint32_t s_st[3];
	const int t = threadIdx.x;
	if (!final) {
		__shared__ uint32_t s_red[3][TH_BS / N2M_WAVE];
		uint32_t omin = 0xffffffffu, omax = 0u, nan = 0u;
		if (t < nrows) {
			omin = rows[3 * t];
			omax = rows[3 * t + 1];
			nan = rows[3 * t + 2];
		}
		omin = wave_min_u32(omin);
		omax = wave_max_u32(omax);
		nan = wave_sum(nan);
		if (lane_id() == 0) {
			s_red[0][wave_id()] = omin;
			s_red[1][wave_id()] = omax;
			s_red[2][wave_id()] = nan;
		}
		__syncthreads();
		if (t == 0) {
			for (int w = 1; w < TH_BS / N2M_WAVE; w++) {
				omin = min(omin, s_red[0][w]);
				omax = max(omax, s_red[1][w]);
				nan += s_red[2][w];
			}
			r->stats[0] = s_st[0] = omin;
			r->stats[1] = s_st[1] = omax;
			r->stats[2] = s_st[2] = nan;
			r->stats[3] = 0u;
			r->par[0] = r->par[1] = 0.0f;
			r->do1001 = 0;
		}
	} else if (t < 3) {
		s_st[t] = r->stats[t];
	}
	__syncthreads();
	const size_t nNan = s_st[2];
	const float mn = ord2f(s_st[0]), mx = ord2f(s_st[1]);
	float pct2 = 0.0f, pct98 = 1.0f;
	if (nvox == nNan) {
		// all NaN: the range keeps its 0..1 defaults
	} else if (mn == mx) {
		pct2 = mn;
		pct98 = mx;
	} else {
		const size_t valid = nvox - nNan;
		const size_t n2pct = (size_t)round(valid * 0.02);
		if (n2pct < 1 || valid < 100) {
			pct2 = mn;
			pct98 = mx;
		} else { // the same for every thread
			const float scl = (kBins - 1) / (mx - mn);
			if (!final) {
				if (t == 0) {
					r->do1001 = 1;
					r->par[0] = mn;
					r->par[1] = scl;
				}
				return;
			}
			// robust_walk() over the summed bins: lo is the first bin whose
			// count from below reaches n2pct, hi the last from above
			__shared__ uint32_t s_h[TH_BS];
			__shared__ unsigned long long s_wave[TH_BS / N2M_WAVE];
			__shared__ int s_lo, s_hi;
			uint32_t c = 0;
			if (t < kBins)
#pragma unroll 32
				for (int i = 0; i < nrows; i++)
					c += rows[(size_t)kBins * i + t];
			s_h[t] = c;
			if (t == 0) {
				s_lo = 0;
				s_hi = kBins - 1;
			}
			// 64-bit sums; the bins and the NaN count themselves have 32 bits, so
			// none of them may reach 2^32 voxels
			unsigned long long upto = c;
#pragma unroll
			for (int d = 1; d < N2M_WAVE; d <<= 1) {
				const unsigned long long o = __shfl_up(upto, d);
				upto += lane_id() >= d ? o : 0ull;
			}
			if (lane_id() == N2M_WAVE - 1)
				s_wave[wave_id()] = upto;
			__syncthreads();
			unsigned long long all = 0;
			for (int w = 0; w < TH_BS / N2M_WAVE; w++) {
				upto += w < wave_id() ? s_wave[w] : 0ull;
				all += s_wave[w];
			}
			const unsigned long long before = upto - c;
			if (upto >= n2pct && before < n2pct)
				s_lo = t;
			if (t < kBins && all - before >= n2pct && all - upto < n2pct)
				s_hi = t;
			__syncthreads();
			if (t == 0) {
				int lo = s_lo, hi = s_hi;
				if (lo == hi) // both move outwards to the next bins in use
					robust_walk(s_h, kBins, n2pct, &lo, &hi);
				pct2 = (lo) / scl + mn;
				pct98 = (hi) / scl + mn;
			}
		}
	}
	if (final && t == 0) {
		const int nBin = 256;
		r->par[2] = pct2;
		r->par[3] = (nBin - 1) / (pct98 - pct2);
	}
}

// work: the rows of a pass, then (once the last histogram is summed) the
// Liao table and, after it, its running sums
static_assert(N2M_THR_WORK >= (size_t)TH_ROWS * TH_BINS * sizeof(uint32_t), "the rows of the longest pass fit");
static_assert((size_t)256 * 256 * 8 >= (size_t)TH_ROWS * 256 * 4, "the sums are not among the rows they come from");
static_assert((size_t)(256 + 2) * 256 * 8 <= N2M_THR_WORK, "table and sums fit");

void launch_threshold_chain(const float *img, size_t nvox, ThrRecord *rec, void *work, bool need5, hipStream_t s)
{
	const unsigned nr = thr_rows(nvox);
	uint32_t *rows = (uint32_t *)work;
	double *PT = (double *)work, *sums = PT + 256 * 256;
	hipLaunchKernelGGL(k_hist_range, dim3(nr), dim3(TH_BS), 0, s, img, nvox, rows);
	hipLaunchKernelGGL(k_thr_range, dim3(1), dim3(TH_BS), 0, s, rec, (const uint32_t *)rows, (int)nr, nvox, 0);
	hipLaunchKernelGGL(k_hist_bins, dim3(nr), dim3(TH_BS), 0, s, img, nvox, (const float *)rec->par,
	                   (const int32_t *)&rec->do1001, TH_BINS, rows);
	hipLaunchKernelGGL(k_thr_range, dim3(1), dim3(TH_BS), 0, s, rec, (const uint32_t *)rows, (int)nr, nvox, 1);
	hipLaunchKernelGGL(k_hist_bins, dim3(nr), dim3(TH_BS), 0, s, img, nvox, (const float *)(rec->par + 2),
	                   (const int32_t *)nullptr, 256, rows);
	hipLaunchKernelGGL(k_otsu_sums, dim3(1), dim3(TH_BS), 0, s, (const uint32_t *)rows, (int)nr, rec->h256, sums);
	hipLaunchKernelGGL(k_otsu_table, dim3(256), dim3(256), 0, s, (const double *)sums, PT, rec->probe);
	if (need5)
		hipLaunchKernelGGL(k_otsu3, dim3(256 - 3), dim3(256 * OT_Q), 0, s, (const double *)PT, 1, 256, 256, rec->bv, rec->bm,
		                   rec->bh);
}


// ---------------------------------------------------------------------------
// Raw NIfTI voxels to the FP32 working volume, src/nii2mesh.c:155-172:
// out = (raw * slope) + inter in float (two roundings), for uint8, int16,
// uint16 and float32 data.
// ---------------------------------------------------------------------------
// Bound by memory.  VEC: 16-byte stores and loads of DEC_VPT raw voxels at a time (raw and out
// aligned to that); the last n % DEC_VPT voxels one by one.
constexpr int DEC_VPT = 8;
template <typename T, bool VEC>
__global__ void __launch_bounds__(256)
k_decode(const T *__restrict__ raw, size_t n, float slope, float inter, float *__restrict__ out)
{
	const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
	size_t done = 0;
	if (VEC) {
		struct alignas(DEC_VPT * sizeof(T) < 16 ? DEC_VPT * sizeof(T) : 16) Pack {
			T v[DEC_VPT];
		};
		const size_t np = n / DEC_VPT;
		for (size_t i = tid; i < np; i += stride) {
			const Pack p = reinterpret_cast<const Pack *>(raw)[i];
			float f[DEC_VPT];
#pragma unroll
			for (int k = 0; k < DEC_VPT; k++) {
				const float v = (float)p.v[k] * slope;
				f[k] = v + inter;
			}
			float4 *o = reinterpret_cast<float4 *>(out) + i * (DEC_VPT / 4);
#pragma unroll
			for (int k = 0; k < DEC_VPT / 4; k++)
				o[k] = make_float4(f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]);
		}
		done = np * DEC_VPT;
	}
	for (size_t i = done + tid; i < n; i += stride) {
		const float v = (float)raw[i] * slope;
		out[i] = v + inter;
	}
}

template <typename T>
static void decode_launch(const void *raw, size_t n, float slope, float inter, float *out, hipStream_t s)
{
	const uintptr_t at = DEC_VPT * sizeof(T) < 16 ? DEC_VPT * sizeof(T) : 16;
	const bool vec = ((uintptr_t)raw % at) == 0 && ((uintptr_t)out & 15u) == 0;
	const size_t per = 256 * (size_t)(vec ? DEC_VPT : 4);
	size_t b = (n + per - 1) / per;
	b = b > 8192 ? 8192 : (b < 1 ? 1 : b);
	const auto k = vec ? k_decode<T, true> : k_decode<T, false>;
	hipLaunchKernelGGL(k, dim3((unsigned)b), dim3(256), 0, s, (const T *)raw, n, slope, inter, out);
}

int launch_decode(const void *raw, int datatype, size_t n, float slope, float inter, float *out, hipStream_t s)
{
	switch (datatype) {
	case 2: // DT_UINT8
		decode_launch<uint8_t>(raw, n, slope, inter, out, s);
		return 0;
	case 4: // DT_INT16
		decode_launch<int16_t>(raw, n, slope, inter, out, s);
		return 0;
	case 512: // DT_UINT16
		decode_launch<uint16_t>(raw, n, slope, inter, out, s);
		return 0;
	case 16: // DT_FLOAT32
		decode_launch<float>(raw, n, slope, inter, out, s);
		return 0;
	}
	return -1;
}

} // namespace n2m
