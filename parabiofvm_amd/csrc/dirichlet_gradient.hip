// Dirichlet conditions and central-difference gradients on gfx950.
#include <algorithm>
#include <type_traits>

#include "bfvm_internal.hpp"

namespace bfvm {

// ------------------------------------------------------------------------------------------------
// Dirichlet — host/dirichlet_solver.cpp:22-144
// ------------------------------------------------------------------------------------------------

// Boundary faces.  One thread per (face voxel, substrate); every voxel on several faces gets the value of the
// last face in the order x-, x+, y-, y+, z-, z+ whose condition is set (host/dirichlet_solver.cpp:91-110),
// so threads that reach the same edge voxel from different faces write the same value.
// Face voxels are enumerated as the two x planes (2*Y*Z), then the two y planes (2*X*Z), then the two z
// planes (2*X*Y) of the axes the mesh has.
template <int K>
__global__ __launch_bounds__(256) void dirichlet_faces_kernel(void* __restrict__ dens, const float* __restrict__ fval,
															  const uint8_t* __restrict__ fcond,
															  const float* __restrict__ scale, int X, int Y, int Z,
															  int S, int dims, int64_t total)
{
	const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (idx >= total)
		return;
	const int s = (int)(idx % S);
	int64_t r = idx / S;
	int x, y, z;
	const int64_t nx = dims >= 1 ? 2 * (int64_t)Y * Z : 0;
	const int64_t ny = dims >= 2 ? 2 * (int64_t)X * Z : 0;
	if (r < nx)
	{
		const int64_t side = r / ((int64_t)Y * Z);
		const int64_t rem = r % ((int64_t)Y * Z);
		x = side ? X - 1 : 0;
		y = (int)(rem % Y);
		z = (int)(rem / Y);
	}
	else if (r < nx + ny)
	{
		r -= nx;
		const int64_t side = r / ((int64_t)X * Z);
		const int64_t rem = r % ((int64_t)X * Z);
		y = side ? Y - 1 : 0;
		x = (int)(rem % X);
		z = (int)(rem / X);
	}
	else
	{
		r -= nx + ny;
		const int64_t side = r / ((int64_t)X * Y);
		const int64_t rem = r % ((int64_t)X * Y);
		z = side ? Z - 1 : 0;
		x = (int)(rem % X);
		y = (int)(rem / X);
	}
	const int coord[3] = { x, y, z };
	const int grid[3] = { X, Y, Z };
	bool set = false;
	float v = 0;
	for (int d = 0; d < dims; d++)
	{
		if (coord[d] == 0 && fcond[(2 * d) * S + s])
		{
			set = true;
			v = fval[(2 * d) * S + s];
		}
		if (coord[d] == grid[d] - 1 && fcond[(2 * d + 1) * S + s])
		{
			set = true;
			v = fval[(2 * d + 1) * S + s];
		}
	}
	if (set)
		dstore<K, 1>(dens, (((int64_t)z * Y + y) * X + x) * S + s, K == store_f32 ? v : v * scale[s]);
}

// Interior list, de-duplicated per voxel at upload (host/dirichlet_solver.cpp:22-44).  One thread per
// (entry, substrate).
template <int K>
__global__ __launch_bounds__(256) void dirichlet_interior_kernel(void* __restrict__ dens,
																 const int64_t* __restrict__ vox,
																 const float* __restrict__ val,
																 const uint8_t* __restrict__ cond,
																 const float* __restrict__ scale, int S,
																 int64_t total)
{
	const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (idx >= total)
		return;
	const int64_t i = idx / S;
	const int s = (int)(idx % S);
	if (cond[idx])
		dstore<K, 1>(dens, vox[i] * S + s, K == store_f32 ? val[idx] : val[idx] * scale[s]);
}

void launch_dirichlet_faces(bfvm_ctx* ctx)
{
	if (!ctx->has_faces)
		return;
	const auto& m = ctx->mesh;
	const int X = m.grid[0], Y = m.grid[1], Z = m.grid[2];
	int64_t faces = 2 * (int64_t)Y * Z;
	if (m.dims >= 2)
		faces += 2 * (int64_t)X * Z;
	if (m.dims >= 3)
		faces += 2 * (int64_t)X * Y;
	const int64_t total = faces * m.S;
	by_storage(ctx->storage, [&](auto k) {
		hipLaunchKernelGGL((dirichlet_faces_kernel<decltype(k)::value>), dim3((unsigned)((total + 255) / 256)),
						   dim3(256), 0, ctx->stream, ctx->dens, ctx->face_val, ctx->face_cond, ctx->dscale, X, Y, Z,
						   m.S, m.dims, total);
	});
	BFVM_HIP(hipGetLastError());
}

void launch_dirichlet_interior(bfvm_ctx* ctx)
{
	if (ctx->n_interior == 0)
		return;
	const int64_t total = ctx->n_interior * ctx->mesh.S;
	by_storage(ctx->storage, [&](auto k) {
		hipLaunchKernelGGL((dirichlet_interior_kernel<decltype(k)::value>), dim3((unsigned)((total + 255) / 256)),
						   dim3(256), 0, ctx->stream, ctx->dens, ctx->int_vox, ctx->int_val, ctx->int_cond, ctx->dscale,
						   ctx->mesh.S, total);
	});
	BFVM_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------------------------------
// gradient — host/gradient_solver.cpp:10-291
// ------------------------------------------------------------------------------------------------
//
// Interior: (d[i+1] - d[i-1]) * (1.f/(2 dx)); borders: (d[1] - d[0]) * (1.f/dx) and (d[n-1] - d[n-2]) * (1.f/dx),
// with the float reciprocals of the reference (host/gradient_solver.cpp:17-18).  Output layout [d][z][y][x][s] in 3-D,
// [y][x][s][d] in 1-D/2-D (src/traits.h:27-33, 55-62, 86-92).

struct gradient_args
{
	float* grad;
	const void* dens;
	const float* inv; // 1 / storage scale of each substrate (16-bit storage)
	int X, Y, Z, S, XS;
	int cols, lanes;		  // columns of a row (4 consecutive positions q = x S + s each); (row band, column) pairs
	int tiles, zchunk, zchunks; // workgroups of a z chunk, planes of a chunk, chunks
	int per_xcd, order;
	float bx, cx, by, cy, bz, cz;
	int64_t VS;
};

// One thread per (voxel, substrate): 1-D meshes, rows shorter than 4 elements or too long for 32-bit row offsets.
template <int K>
__global__ __launch_bounds__(256) void gradient_kernel(gradient_args a, int dims)
{
	const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (idx >= a.VS)
		return;
	const int64_t v = idx / a.S;
	const int x = (int)(v % a.X), y = (int)((v / a.X) % a.Y), z = (int)(v / ((int64_t)a.X * a.Y));
	const float is = K == store_f32 ? 1.f : a.inv[idx % a.S];
	auto p = [&](int64_t o) {
		const float d = dload<K, 1>(a.dens, idx + o);
		return K == store_f32 ? d : d * is;
	};
	auto diff = [&](int i, int n, int64_t stride, float b, float c) {
		const int64_t up = i + 1 < n ? stride : 0, down = i > 0 ? stride : 0;
		return (p(up) - p(-down)) * (up && down ? c : b);
	};
	const int64_t out = dims == 3 ? idx : idx * dims, step = dims == 3 ? a.VS : 1;
	a.grad[out] = diff(x, a.X, a.S, a.bx, a.cx);
	if (dims >= 2)
		a.grad[out + step] = diff(y, a.Y, a.XS, a.by, a.cy);
	if (dims == 3)
		a.grad[out + 2 * step] = diff(z, a.Z, (int64_t)a.Y * a.XS, a.bz, a.cz);
}

constexpr int grad_tile = 256;
constexpr int num_xcds = 8;

template <int K>
struct uvec
{
	using type = typename store_of<K>::elem __attribute__((ext_vector_type(4), aligned(sizeof(typename store_of<K>::elem))));
};
using float4u = float __attribute__((ext_vector_type(4), aligned(4)));

// 2-D and 3-D: one thread per (band of TY rows, column of 4 consecutive row positions), with or without a march over
// the planes of a z chunk (the z - 1, z, z + 1 densities of its rows in registers, the next plane's loads issued before
// this plane's results).  Bound by memory: a 3-D gradient writes 3 floats per density, so what a kernel can lose is
// re-reading densities and the order of its writes.
//  - No condition around a load: rows and planes outside the mesh are clamped into it, so the neighbour that a
//    one-sided difference does not have is the element itself and only the factor differs, and every load of a step is
//    in flight at once.  Loads under a lane's own condition are waited for one by one.
//  - ALIGNED: 4 divides S, a vector is 4 substrates of one voxel; otherwise its positions are of different substrates
//    and voxels, accesses are at element alignment, x = 0 and x = X - 1 are told per position, and a row's last column
//    is moved back to end with the row (it computes 4 positions and stores the ones it owns).
//  - The (band, column) pairs of a plane are numbered through, so short rows fill the waves as long ones do.
// Which of the forms, and the order of the workgroups: gradient_shape_of.
template <int K, int TY, bool ALIGNED, int DIMS, bool MARCH>
__global__ __launch_bounds__(grad_tile) void gradient_field_kernel(gradient_args a)
{
	using vec = typename vec_of<4>::type;
	using elem = typename store_of<K>::elem;
	using raw = std::conditional_t<ALIGNED, typename svec_of<K, 4>::type, typename uvec<K>::type>;
	using out = std::conditional_t<ALIGNED, vec, float4u>;
	// order 0: consecutive (tile, chunk) pairs on one XCD (the dispatcher hands it workgroup b % 8), so that its L2
	// serves the rows and planes where they meet; order 1: the workgroups as they come, all XCDs in one narrow window
	// of each output
	const int b = a.order == 0 ? (int)(blockIdx.x % num_xcds) * a.per_xcd + (int)(blockIdx.x / num_xcds) : (int)blockIdx.x;
	const int zc = b / a.tiles;
	const int id = (b - zc * a.tiles) * grad_tile + threadIdx.x;
	if (id >= a.lanes || zc >= a.zchunks)
		return;
	const int band = id / a.cols, col = id - band * a.cols;
	const int S = a.S, XS = a.XS, Y = a.Y, Z = a.Z;
	const int q = ALIGNED ? col * 4 : min(col * 4, XS - 4);
	const int y0 = band * TY;
	const int64_t plane = (int64_t)Y * XS, lane = (int64_t)y0 * XS + q;
	int row[TY + 2]; // rows y0 - 1 .. y0 + TY, clamped into the mesh, relative to the thread's first element
#pragma unroll
	for (int r = 0; r < TY + 2; r++)
		row[r] = (min(max(y0 + r - 1, 0), Y - 1) - y0) * XS;
	// aligned vectors lie in one voxel: the neighbour in x beyond the mesh is the voxel itself
	const int left = ALIGNED && q < S ? 0 : S, right = ALIGNED && q >= XS - S ? 0 : S;
	vec kx, is = vec(1.f);
#pragma unroll
	for (int c = 0; c < 4; c++)
	{
		kx[c] = q + c < S || q + c >= XS - S ? a.bx : a.cx;
		if constexpr (K != store_f32)
			is[c] = a.inv[(q + c) % S];
	}
	const elem* dens = (const elem*)a.dens + lane;
	auto at = [&](int z) { return dens + (DIMS == 3 ? min(max(z, 0), Z - 1) * plane : 0); };
	auto ld = [&](const elem* p) { return gload((const raw*)p); };
	auto cv = [&](raw r) -> vec {
		if constexpr (K == store_f32)
			return (vec)r;
		else
			return __builtin_convertvector(r, vec) * is;
	};
	// the loads of plane z that do not stay in registers, and plane z + 1
	raw next[TY], lo, hi, xm[TY], xp[TY];
	// unaligned x neighbours of the array's first and last elements: moved into the array, put right by `place`
	const bool first_rows = !ALIGNED && band == 0, last_rows = !ALIGNED && y0 + TY >= Y;
	const int rem = last_rows ? (int)(plane - lane) : 0;
	auto fetch = [&](int z) {
		const elem *p = at(z), *p1 = at(z + 1);
		const bool first = first_rows && (DIMS == 2 || z == 0), last = last_rows && (DIMS == 2 || z == Z - 1);
		lo = ld(p + row[0]);
		hi = ld(p + row[TY + 1]);
#pragma unroll
		for (int r = 0; r < TY; r++)
		{
			const int o = row[r + 1];
			if constexpr (DIMS == 3)
				next[r] = ld(p1 + o);
			xm[r] = ld(p + (first ? max(o - left, -q) : o - left));
			xp[r] = ld(p + (last ? min(o + right, rem - 4) : o + right));
		}
	};
	auto place = [&](vec v, int n, bool up) { // v[c + n] or v[c - n], where that exists
		vec r = v;
#pragma unroll
		for (int c = 0; c < 4; c++)
#pragma unroll
			for (int m = 1; m < 4; m++)
				if (up ? c + m < 4 : c - m >= 0)
					r[c] = n == m ? v[up ? c + m : c - m] : r[c];
		return r;
	};
	const int z0 = zc * a.zchunk, z1 = MARCH ? min(Z, z0 + a.zchunk) : z0 + 1;
	vec zm[TY], c[TY];
	{
		raw r0[TY], r1[TY];
#pragma unroll
		for (int r = 0; r < TY; r++)
		{
			if constexpr (DIMS == 3)
				r0[r] = ld(at(z0 - 1) + row[r + 1]);
			r1[r] = ld(at(z0) + row[r + 1]);
		}
		fetch(z0);
#pragma unroll
		for (int r = 0; r < TY; r++)
		{
			if constexpr (DIMS == 3)
				zm[r] = cv(r0[r]);
			c[r] = cv(r1[r]);
		}
	}
	const int own = XS - col * 4; // below 4: the positions of a moved-back column
	for (int z = z0; z < z1; z++)
	{
		vec zp[TY], vm[TY], vp[TY];
#pragma unroll
		for (int r = 0; r < TY; r++)
		{
			if constexpr (DIMS == 3)
				zp[r] = cv(next[r]);
			vm[r] = cv(xm[r]);
			vp[r] = cv(xp[r]);
		}
		const vec below = cv(lo), above = cv(hi);
		if constexpr (!ALIGNED)
		{
			if (first_rows && (DIMS == 2 || z == 0))
#pragma unroll
				for (int r = 0; r < TY; r++)
					vm[r] = place(vm[r], max(S - q - row[r + 1], 0), false);
			if (last_rows && (DIMS == 2 || z == Z - 1))
#pragma unroll
				for (int r = 0; r < TY; r++)
					vp[r] = place(vp[r], max(row[r + 1] + S + 4 - rem, 0), true);
		}
		if (MARCH && z + 1 < z1)
			fetch(z + 1);
		const float kz = z == 0 || z == Z - 1 ? a.bz : a.cz;
#pragma unroll
		for (int r = 0; r < TY; r++)
		{
			const int y = y0 + r;
			vec gx, gy, gz;
			if constexpr (ALIGNED)
				gx = (vp[r] - vm[r]) * kx;
			else
#pragma unroll
				for (int i = 0; i < 4; i++)
					gx[i] = ((q + i >= XS - S ? c[r][i] : vp[r][i]) - (q + i < S ? c[r][i] : vm[r][i])) * kx[i];
			const vec ym = r == 0 ? below : c[r - 1 < 0 ? 0 : r - 1];
			const vec yp = r == TY - 1 ? above : c[r + 1 < TY ? r + 1 : r];
			gy = (yp - ym) * (y == 0 || y == Y - 1 ? a.by : a.cy);
			if constexpr (DIMS == 3)
				gz = (zp[r] - zm[r]) * kz;
			if (y >= Y)
				break;
			if constexpr (DIMS == 3)
			{
				// streaming outputs: non-temporal stores leave the caches to the densities (400^3 x 8 FP32 1.51 ->
				// 1.39 ms, 177x181x179 x 7 0.135 -> 0.123 ms)
				float* g = a.grad + z * plane + lane + row[r + 1];
				if (ALIGNED || own >= 4)
				{
					__builtin_nontemporal_store((out)gx, (out*)g);
					__builtin_nontemporal_store((out)gy, (out*)(g + a.VS));
					__builtin_nontemporal_store((out)gz, (out*)(g + 2 * a.VS));
				}
				else
#pragma unroll
					for (int i = 1; i < 4; i++)
						if (i >= 4 - own)
						{
							__builtin_nontemporal_store(gx[i], g + i);
							__builtin_nontemporal_store(gy[i], g + i + a.VS);
							__builtin_nontemporal_store(gz[i], g + i + 2 * a.VS);
						}
			}
			else
			{
				float* g = a.grad + 2 * (lane + row[r + 1]);
				const vec g0 { gx[0], gy[0], gx[1], gy[1] }, g1 { gx[2], gy[2], gx[3], gy[3] };
				if (ALIGNED || own >= 4)
				{
					gstore((out*)g, (out)g0);
					gstore((out*)(g + 4), (out)g1);
				}
				else
#pragma unroll
					for (int i = 1; i < 4; i++)
						if (i >= 4 - own)
						{
							gstore(g + 2 * i, gx[i]);
							gstore(g + 2 * i + 1, gy[i]);
						}
			}
		}
		if constexpr (MARCH)
#pragma unroll
			for (int r = 0; r < TY; r++)
			{
				zm[r] = c[r];
				c[r] = zp[r];
			}
	}
}

// Calibration kernel: float4 copy of n4 16-byte elements.  Its bandwidth is the practical ceiling the
// solver kernels are compared against, and its counter readings scale the traffic counters.
__global__ __launch_bounds__(256) void copy_kernel(float4* __restrict__ dst, const float4* __restrict__ src,
												   int64_t n4)
{
	const int64_t stride = (int64_t)gridDim.x * blockDim.x;
	for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride)
		dst[i] = src[i];
}

void launch_copy(bfvm_ctx* ctx)
{
	const int64_t bytes = (int64_t)ctx->mesh.V * ctx->mesh.S * (ctx->storage == BFVM_STORAGE_F32 ? 4 : 2);
	const int64_t n4 = bytes / 16;
	if (n4 == 0)
		return;
	// one 16-byte element per thread in 256-thread workgroups, one pass over the array (up to 2^30 workgroups):
	// the launch shape that moved the most bytes per second on MI355X (6.1 TB/s against 5.2-5.8 TB/s for
	// persistent grid-stride launches and 5.8 TB/s for 1024-thread workgroups)
	const int64_t blocks = std::min<int64_t>(int64_t(1) << 30, (n4 + 255) / 256);
	hipLaunchKernelGGL(copy_kernel, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, (float4*)ctx->grad,
					   (const float4*)ctx->dens, n4);
	BFVM_HIP(hipGetLastError());
}

// The form of a 3-D gradient and its tiling.
//  - Densities that fit in the Infinity Cache (256 MiB; in FP32 up to 15/16 of it): 2 rows per thread, no march, order
//    0.  The neighbouring planes are read from the caches, and the most workgroups are in flight.  2 rows / 8 rows with
//    march, us: 60x50x40 x 4 FP32 3.6 / 9.5, 200^3 x 4 FP32 71 / 98, 177x181x179 x 7 FP32 123 / 160, FP16 131 / 157,
//    256^3 x 8 FP16 256 / 298.
//  - Larger: 8 rows per thread marching over 3 planes, in plane order.  One march step loads 10 rows for 8, the first
//    planes of a chunk are the last ones of the chunk before, still cached, and the three outputs are written in narrow
//    windows; longer chunks spread the windows.  2 rows / 8 rows: 256^3 x 5 FP32 328 / 238, 400^3 x 8 FP32 1735 / 1387
//    (5.9 TB/s; 8 planes 1480, order 0 1570), FP16 1843 / 1198 (6.0 TB/s), 320^3 x 8 FP16 945 / 640, 256^3 x 16 FP16
//    957 / 689.
//    The line depends on what the caches hold: as a step leaves the densities, or read over and over, 2 rows are ahead up
//    to the cache's size (4, 5, 8 substrates at 0.97 of it, FP32 184 238 183 / 226 255 207, FP16 371 357 351 / 441 397
//    408; at 1.05 FP32 281 277 249 / 205 263 222); on densities that other work has displaced the march is ahead from
//    0.8 of it (at 0.97 FP32 270 297 265 / 241 261 208, FP16 466 483 468 / 420 411 425; 320^3 x 8 FP16 741 by the
//    march).  15/16 in FP32, whose loss is the larger on that side, is between the two.
//  - With workgroup counts or layouts of the caller or the autotuner: 8 rows (stacked) or 4 rows, marching.
struct gradient_shape
{
	int rows, zchunk, order;
};
static gradient_shape gradient_shape_of(const bfvm_ctx* ctx, int64_t bytes)
{
	const auto& m = ctx->mesh;
	if (ctx->gradient_groups == 0 && !ctx->gradient_stacked && ctx->gradient_order == 0)
	{
		const int64_t cache = ((int64_t)256 << 20) / 16 * (ctx->storage == BFVM_STORAGE_F32 ? 15 : 16);
		return bytes <= cache ? gradient_shape { 2, 1, 0 } : gradient_shape { 8, 3, 1 };
	}
	const int rows = ctx->gradient_stacked ? 8 : 4;
	const int64_t target = ctx->gradient_groups > 0 ? ctx->gradient_groups : 16384;
	const int64_t lanes = ((int64_t)m.grid[0] * m.S + 3) / 4 * ((m.grid[1] + rows - 1) / rows);
	const int64_t tiles = (lanes + grad_tile - 1) / grad_tile;
	const int chunks = (int)std::max<int64_t>(1, std::min<int64_t>(m.grid[2], (target + tiles - 1) / tiles));
	return { rows, (m.grid[2] + chunks - 1) / chunks, ctx->gradient_order };
}

template <int K, bool ALIGNED>
static void launch_gradient_field(const bfvm_ctx* ctx, gradient_args a, int rows)
{
	const int64_t workgroups = a.order == 0 ? (int64_t)a.per_xcd * num_xcds : (int64_t)a.tiles * a.zchunks;
	auto kernel = ctx->mesh.dims == 2 ? gradient_field_kernel<K, 2, ALIGNED, 2, false>
				  : rows == 2		  ? gradient_field_kernel<K, 2, ALIGNED, 3, false>
				  : rows == 4		  ? gradient_field_kernel<K, 4, ALIGNED, 3, true>
									  : gradient_field_kernel<K, 8, ALIGNED, 3, true>;
	hipLaunchKernelGGL(kernel, dim3((unsigned)workgroups), dim3(grad_tile), 0, ctx->stream, a);
}

void launch_gradient(bfvm_ctx* ctx)
{
	const auto& m = ctx->mesh;
	gradient_args a {};
	a.grad = ctx->grad;
	a.dens = ctx->dens;
	a.inv = ctx->dinv;
	a.X = m.grid[0];
	a.Y = m.grid[1];
	a.Z = m.grid[2];
	a.S = m.S;
	a.XS = m.grid[0] * m.S;
	a.VS = (int64_t)m.V * m.S;
	a.bx = 1.f / m.vs[0];
	a.cx = 1.f / (m.vs[0] * 2);
	if (m.dims >= 2)
	{
		a.by = 1.f / m.vs[1];
		a.cy = 1.f / (m.vs[1] * 2);
	}
	if (m.dims == 3)
	{
		a.bz = 1.f / m.vs[2];
		a.cz = 1.f / (m.vs[2] * 2);
	}
	const gradient_shape shape = m.dims == 3 ? gradient_shape_of(ctx, a.VS * (int64_t)storage_bytes(ctx->storage))
											 : gradient_shape { 2, 1, 0 };
	const int64_t lanes = ((int64_t)a.XS + 3) / 4 * ((a.Y + shape.rows - 1) / shape.rows);
	const int64_t tiles = (lanes + grad_tile - 1) / grad_tile, chunks = (a.Z + shape.zchunk - 1) / shape.zchunk;
	// row offsets within a thread's rows, lanes and workgroups are 32-bit
	const bool field = m.dims >= 2 && a.XS >= 4 && a.XS < 1 << 27 && lanes + grad_tile < (int64_t)1 << 31 &&
					   tiles * chunks + num_xcds < (int64_t)1 << 31;
	by_storage(ctx->storage, [&](auto k) {
		constexpr int K = decltype(k)::value;
		if (!field)
		{
			hipLaunchKernelGGL(gradient_kernel<K>, dim3((unsigned)((a.VS + 255) / 256)), dim3(256), 0, ctx->stream, a,
							   m.dims);
			return;
		}
		a.cols = (a.XS + 3) / 4;
		a.lanes = (int)lanes;
		a.tiles = (int)tiles;
		a.zchunk = shape.zchunk;
		a.zchunks = (int)chunks;
		a.per_xcd = (int)((tiles * chunks + num_xcds - 1) / num_xcds);
		a.order = shape.order;
		if (m.S % 4 == 0)
			launch_gradient_field<K, true>(ctx, a, shape.rows);
		else
			launch_gradient_field<K, false>(ctx, a, shape.rows);
	});
	BFVM_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------------------------------
// FP32 <-> storage conversions (uploads and downloads of the densities)
// ------------------------------------------------------------------------------------------------

template <int K>
__global__ __launch_bounds__(256) void pack_kernel(void* __restrict__ dens, const float* __restrict__ src,
												   const float* __restrict__ scale, int S, int64_t offset, int64_t n)
{
	const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const int s = (int)((offset + i) % S);
	dstore<K, 1>(dens, offset + i, src[i] * scale[s]);
}

template <int K>
__global__ __launch_bounds__(256) void unpack_kernel(float* __restrict__ dst, const void* __restrict__ dens,
													 const float* __restrict__ inv, int S, int64_t offset, int64_t n)
{
	const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const int s = (int)((offset + i) % S);
	dst[i] = dload<K, 1>(dens, offset + i) * inv[s];
}

// per-substrate max |x| as the bit pattern of a non-negative float (which orders like an unsigned integer)
__global__ __launch_bounds__(256) void max_abs_kernel(const float* __restrict__ src, int S, int64_t n,
													  unsigned* __restrict__ out)
{
	const int64_t stride = (int64_t)gridDim.x * blockDim.x;
	for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
	{
		const float a = fabsf(src[i]);
		if (a > 0.f && a <= 3.4e38f)
			atomicMax(&out[i % S], __float_as_uint(a));
	}
}

// FP16 storage: stored values of substrate s times factor[s] (a power of two, so exact while the result stays
// normal); grid-stride over the whole densities array
__global__ __launch_bounds__(256) void rescale_f16_kernel(_Float16* __restrict__ dens, const float* __restrict__ factor,
														  int S, int64_t n)
{
	const int64_t stride = (int64_t)gridDim.x * blockDim.x;
	for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
		dens[i] = (_Float16)((float)dens[i] * factor[i % S]);
}

void launch_rescale_f16(bfvm_ctx* ctx, const float* factor, hipStream_t stream)
{
	const int64_t n = (int64_t)ctx->mesh.V * ctx->mesh.S;
	const unsigned blocks = (unsigned)std::min<int64_t>(8192, (n + 255) / 256);
	hipLaunchKernelGGL(rescale_f16_kernel, dim3(blocks), dim3(256), 0, stream, (_Float16*)ctx->dens, factor,
					   ctx->mesh.S, n);
	BFVM_HIP(hipGetLastError());
}

__global__ void advance_rounding_kernel(unsigned* counter)
{
	if (threadIdx.x == 0)
		*counter = *counter + 1;
}

void launch_advance_rounding(bfvm_ctx* ctx)
{
	hipLaunchKernelGGL(advance_rounding_kernel, dim3(1), dim3(64), 0, ctx->stream, ctx->rounding_step);
	BFVM_HIP(hipGetLastError());
}

void launch_pack(bfvm_ctx* ctx, const float* src, int64_t offset, int64_t n)
{
	by_storage(ctx->storage, [&](auto k) {
		hipLaunchKernelGGL((pack_kernel<decltype(k)::value>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
						   ctx->stream, ctx->dens, src, ctx->dscale, ctx->mesh.S, offset, n);
	});
	BFVM_HIP(hipGetLastError());
}

void launch_unpack(bfvm_ctx* ctx, float* dst, int64_t offset, int64_t n)
{
	by_storage(ctx->storage, [&](auto k) {
		hipLaunchKernelGGL((unpack_kernel<decltype(k)::value>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
						   ctx->stream, dst, ctx->dens, ctx->dinv, ctx->mesh.S, offset, n);
	});
	BFVM_HIP(hipGetLastError());
}

void launch_max_abs(bfvm_ctx* ctx, const float* src, int64_t n, unsigned* out)
{
	hipLaunchKernelGGL(max_abs_kernel, dim3(4096), dim3(256), 0, ctx->stream, src, ctx->mesh.S, n, out);
	BFVM_HIP(hipGetLastError());
}

} // namespace bfvm
