// The x/y/z sweeps as two-sided recursive filters on gfx950.
//
// The system of a line (diffusion.hip) is Toeplitz up to its end rows: with a = dt*D/dx^2 and B = 1 +
// decay*dt/dims + 2a, the interior rows are -a x_{i-1} + B x_i - a x_{i+1} = d_i, and the end rows, whose diagonal
// is B - a, are the interior row with a ghost x_{-1} = x_0 (x_n = x_{n-1}): zero flux, i.e. the line mirrored about
// its ends.  On the mirrored infinite line the matrix factors exactly into two first-order recursions with one
// constant, mu = 2a / (B + sqrt(B^2 - 4a^2)) (the smaller root of a mu^2 - B mu + a = 0, 0 <= mu < 1):
//   u_j = s d_j + mu u_{j-1},   x_j = u_j + mu x_{j+1},   s = (1 - mu)^2 / (1 + decay*dt/dims)
// (s applied to d: nothing on the way exceeds the densities, where it applied to x would have a factor of up to 14).  The
// same solution as the Thomas algorithm's (host/diffusion_solver.cpp:72-142, 297-480), with constants instead of a table
// entry per element: 5 operations per element and no table reads.
// Every term is positive for positive densities, so rounding errors do not amplify, and s is chosen from the rounded mu so
// that a constant field keeps its exact gain.  What the rounding of mu does cost is the distance over which a local
// source decays: a relative error of up to 2^-25 / (mu |ln mu|) of it, which grows with a (filter_coefficients_ok).
//
// A line is split into blocks of m elements held in the registers of one lane each.  Per block: f = sum mu^{m-1-j} s d_j
// and e = sum mu^j s d_j (the block's contribution to everything right and left of it), one two-sided scan of
// (f, e) over the line's blocks (factor W = mu^m per block; lane shuffles within a wave, one LDS exchange where a
// line takes several waves), the mirror images at both ends in closed form, then the two recursions started with
// the exact values of the neighbouring blocks.  Small workgroups (the waves of one line group, 1 to 8) with at most
// one barrier: the groups of a CU drift apart and keep loads, arithmetic and stores in flight at the same time.
//   scan:  U_k = sum_{k'<k} W^{k-1-k'} f_{k'},  T_k = sum_{k'>=k} W^{k'-k} e_{k'}
//   line:  E = T_0, F = f_last + mu^{mlast} U_last (sums of s d_j weighted by the distance to the first / last element)
//   ends:  u_{-1} = (E + mu^n F) / (1 - mu^{2n}),  z_n = (F + mu^n E) / (1 - mu^{2n})
//   block: u_{start-1} = U_k + mu^{m k} u_{-1},  Z = T_{k+1} + mu^{n - min(n, m(k+1))} z_n,
//          x_{end+1} = (mu u_end + Z) / (1 - mu^2)
#include <algorithm>
#include <cmath>

#include "bfvm_internal.hpp"

namespace bfvm {

// Coefficient table of one axis, rows of S floats (powers of the rounded mu, computed in FP64).  A wave holds `kw`
// blocks of a line; blocks rows each of mu^{m k} / (1 - mu^{2n}) and mu^{n - min(n, m(k+1))} / (1 - mu^{2n}) and kw
// rows of mu^{m i} follow the single rows.  A workgroup keeps the table in LDS: held in registers, the 12 vectors a
// lane needs cost it a wave per SIMD.
enum filter_row
{
	fr_mu,
	fr_s,	   // factor of the densities
	fr_inv1,   // 1 / (1 - mu^2)
	fr_mun,	   // mu^n
	fr_w,	   // W = mu^m
	fr_mulast, // mu^mlast
	fr_wk,	   // W^kw: one wave's blocks
	fr_flast,  // mu^mlast W^i, i = the last block's index within its wave
	fr_min,	   // this axis's Dirichlet faces: value and condition (1 or 0) at the line's first and last element
	fr_min_on,
	fr_max,
	fr_max_on,
	fr_ends
};

__global__ void filter_coefficients_kernel(float* __restrict__ tab, const float* __restrict__ D,
										   const float* __restrict__ decay, const float* __restrict__ fval,
										   const uint8_t* __restrict__ fcond, float dt, int shape, int dims, int n,
										   int S, int m, int blocks, int kw)
{
	const int s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= S)
		return;
	const double a = (double)dt * (double)D[s] / ((double)shape * (double)shape);
	const double lam = 1.0 + (double)decay[s] * (double)dt / dims; // B - 2a
	const float muf = (float)(2.0 * a / (lam + 2.0 * a + sqrt(lam * (lam + 4.0 * a))));
	const double mu = muf;
	auto row = [&](int r, double v) { tab[(size_t)r * S + s] = (float)v; };
	const int mlast = n - (blocks - 1) * m;
	const double iden = 1.0 / (1.0 - pow(mu, 2.0 * n));
	row(fr_mu, mu);
	row(fr_s, (1.0 - mu) * (1.0 - mu) / lam);
	row(fr_inv1, 1.0 / (1.0 - mu * mu));
	row(fr_mun, pow(mu, (double)n));
	row(fr_w, pow(mu, (double)m));
	row(fr_mulast, pow(mu, (double)mlast));
	row(fr_wk, pow(mu, (double)m * kw));
	row(fr_flast, pow(mu, (double)mlast + (double)m * ((blocks - 1) % kw)));
	// fval, fcond: [2][S] of this axis
	row(fr_min, fval[s]);
	row(fr_min_on, fcond[s] ? 1.0 : 0.0);
	row(fr_max, fval[S + s]);
	row(fr_max_on, fcond[S + s] ? 1.0 : 0.0);
	for (int k = 0; k < blocks; k++)
	{
		row(fr_ends + k, pow(mu, (double)m * k) * iden);
		row(fr_ends + blocks + k, pow(mu, (double)(n - min(n, m * (k + 1)))) * iden);
	}
	for (int i = 0; i < kw; i++)
		row(fr_ends + 2 * blocks + i, pow(mu, (double)m * i));
}

// One axis of one instance, as launched.
struct filter_args
{
	void* data;
	const float* scale;		  // [S] storage scale (16-bit forms)
	const unsigned* rounding; // step counter keying the stochastic rounding (16-bit forms)
	const float* fval;		  // Dirichlet faces (null: none)
	const uint8_t* fcond;
	const float* tab;
	int grid[3];
	int S, dims, axis;
	int m, blocks, mlast, kw; // block length, blocks of a line, elements of the last block, blocks per wave
	int64_t tasks;			  // line groups, one per workgroup pass
	int64_t stride;			  // elements between neighbours of a line
	// a task is 1 << clog columns of 4 consecutive elements; columns run over ranges of row_elems elements, outer_stride
	// apart (x: the S elements of a voxel, one range per row; y: the XS elements of a plane's rows, one range per z; z:
	// the whole plane, one range)
	int clog;
	uint32_t columns, row_columns;
	int64_t row_elems, outer_stride;
	uint32_t row_mul, s_mul, x_mul; // fdiv pairs of row_columns, S and X (x axis: Y)
	int row_shift, s_shift, x_shift;
	// staged x rows: a task is `rows` rows of XS elements in the workgroup's LDS; lines_pass lines at a time in each wave
	// (kw == blocks) or in all of them
	int rows, lines_pass, passes, staged;
	int64_t total_rows;
	int table_floats;			// floats of the table; in LDS, the storage scales [S] follow (16-bit forms)
	int exchange_at, rows_at; // LDS offsets in bytes of the exchange area and the staged rows
};

// value of lane `src` (any lane of the wave that runs this code)
template <int V>
__device__ __forceinline__ typename vec_of<V>::type lane_vec(typename vec_of<V>::type v, int src)
{
	typename vec_of<V>::type r;
#pragma unroll
	for (int c = 0; c < V; c++)
		set_comp(r, c, __int_as_float(__builtin_amdgcn_ds_bpermute(src << 2, __float_as_int(comp(v, c)))));
	return r;
}

// Values the compiler must take as new: without, everything that depends only on the thread and the mesh (an address
// for each of the M elements, several times over) is computed once before the task loop and held in registers.
__device__ __forceinline__ int fresh_lane_value(int x)
{
	asm volatile("" : "+v"(x));
	return x;
}
__device__ __forceinline__ int fresh_uniform(int x)
{
	x = __builtin_amdgcn_readfirstlane(x);
	asm volatile("" : "+s"(x));
	return x;
}
__device__ __forceinline__ int64_t fresh_uniform(int64_t x)
{
	const uint32_t lo = (uint32_t)fresh_uniform((int)(uint32_t)x), hi = (uint32_t)fresh_uniform((int)(x >> 32));
	return (int64_t)((uint64_t)hi << 32 | lo);
}

// Where a lane's block stands: block k = 0..last of its line, index i = 0..kw-1 among the blocks of its wave (`dist`
// lanes apart), wave 0..waves-1 of the line; `slot` numbers the lines of the workgroup and `slots` counts them.
struct filter_place
{
	int k, last, i, kw, wave, waves, lane, dist, slot, slots;
	bool active;
};

// Elements of a block that every lane has: all of them (FULL), else at least half (choose_filter sees to it).  The
// others are there where j < mk, by selects: branches around single loads or operations made the compiler wait for
// each load where it was issued.
template <int M, bool FULL>
constexpr int sure() { return FULL ? M : M / 2; }

// The filter on one block v[0..mk), mk = M except in the last block of a line (not FULL), the rest of its v zero on
// entry.  store(j, x) runs in descending j < mk, in active lanes.  `sh`: [2][waves][slots] vectors and
// [slots] more, exchanged once where a line takes several waves (then every thread of the workgroup comes here).
template <int M, bool FULL, int V, typename Row, typename Store>
__device__ __forceinline__ void filter_line(typename vec_of<V>::type (&v)[M], Row&& row, int mk, int blocks,
											const filter_place& at, typename vec_of<V>::type* sh, Store&& store)
{
	// held to a tolerance, not to the reference's operation order: multiply-adds fuse
#pragma clang fp contract(fast)
	using vec = typename vec_of<V>::type;
	constexpr int N = sure<M, FULL>();
	auto has = [&](int j) { return j < N || j < mk; };
	const vec mu = row(fr_mu);
	vec f = v[0], e = v[M - 1];
#pragma unroll
	for (int j = 1; j < M; j++)
		f = has(j) ? v[j] + mu * f : f;
#pragma unroll
	for (int j = M - 2; j >= 0; j--)
		e = v[j] + mu * e;
	// scan over the blocks of this wave; selects, not products with zero: lanes of other lines may hold anything
	vec w = row(fr_w), sx = f, tx = e;
	const int upto = min(at.kw - 1, at.last - (at.k - at.i)); // index of the line's last block in this wave
#pragma unroll 1
	for (int d = 1; d < at.kw && d <= at.last; d <<= 1)
	{
		const vec a = lane_vec<V>(sx, at.lane - d * at.dist), b = lane_vec<V>(tx, at.lane + d * at.dist);
		sx = at.i >= d ? sx + w * a : sx;
		tx = at.i + d <= upto ? tx + w * b : tx;
		w = w * w;
	}
	vec u = lane_vec<V>(sx, at.lane - at.dist), z = lane_vec<V>(tx, at.lane + at.dist);
	u = at.i > 0 ? u : vec(0.f);
	z = at.i < upto ? z : vec(0.f);
	vec E, F;
	if (at.waves == 1)
	{
		const int lane0 = at.lane - at.i * at.dist;
		E = lane_vec<V>(tx, lane0);
		F = lane_vec<V>(f + row(fr_mulast) * u, lane0 + at.last * at.dist);
	}
	else
	{
		vec* shs = sh + at.wave * at.slots + at.slot;
		vec* sht = shs + at.waves * at.slots;
		if (at.active)
		{
			if (at.i == at.kw - 1)
				*shs = sx;
			if (at.i == 0)
				*sht = tx;
			if (at.k == at.last)
				sh[2 * at.waves * at.slots + at.slot] = f + row(fr_mulast) * u;
		}
		__syncthreads();
		const vec wk = row(fr_wk);
		vec ul = vec(0.f), tr = vec(0.f), ulast = vec(0.f); // carried into this wave from the left, the right; last wave
		E = vec(0.f);
#pragma unroll 1
		for (int o = 0; o < at.waves - 1; o++)
		{
			ulast = sh[o * at.slots + at.slot] + wk * ulast;
			if (o < at.wave)
				ul = ulast;
		}
#pragma unroll 1
		for (int o = at.waves - 1; o >= 0; o--)
		{
			E = sh[(at.waves + o) * at.slots + at.slot] + wk * E;
			if (o == at.wave + 1)
				tr = E;
		}
		F = sh[2 * at.waves * at.slots + at.slot] + row(fr_flast) * ulast;
		u = u + row(fr_ends + 2 * blocks + at.i) * ul;
		z = z + row(fr_ends + 2 * blocks + at.kw - 1 - at.i) * tr;
	}
	const vec mun = row(fr_mun);
	const int kt = min(at.k, at.last); // inactive lanes read a row that is there
	u = u + row(fr_ends + kt) * (E + mun * F);
	z = z + row(fr_ends + blocks + kt) * (F + mun * E);
#pragma unroll
	for (int j = 0; j < M; j++)
	{
		u = has(j) ? v[j] + mu * u : u;
		v[j] = u;
	}
	vec x = (mu * u + z) * row(fr_inv1);
	if (at.active)
	{
#pragma unroll
		for (int j = M - 1; j >= 0; j--)
		{
			x = has(j) ? v[j] + mu * x : x;
			if (has(j))
				store(j, x);
		}
	}
}

// The table (and the storage scales) into LDS, in two halves so that the loads fly with the data's: table_load
// before the data's loads, table_store after them.  Tables of more than table_regs floats per thread continue in
// the second half.
constexpr int table_regs = 4;
template <int K>
__device__ __forceinline__ void table_load(const filter_args& a, float (&t)[table_regs])
{
	const int total = a.table_floats + (K == store_f32 ? 0 : a.S);
#pragma unroll
	for (int j = 0; j < table_regs; j++)
	{
		const int i = threadIdx.x + j * blockDim.x;
		if (i < a.table_floats)
			t[j] = gload(a.tab + i);
		else if (i < total)
			t[j] = gload(a.scale + i - a.table_floats);
	}
}
template <int K>
__device__ __forceinline__ void table_store(const filter_args& a, const float (&t)[table_regs], float* lt)
{
	const int total = a.table_floats + (K == store_f32 ? 0 : a.S);
#pragma unroll
	for (int j = 0; j < table_regs; j++)
	{
		const int i = threadIdx.x + j * blockDim.x;
		if (i < total)
			lt[i] = t[j];
	}
	for (int i = threadIdx.x + table_regs * blockDim.x; i < total; i += blockDim.x)
		lt[i] = i < a.table_floats ? gload(a.tab + i) : gload(a.scale + i - a.table_floats);
}

// Order within a workgroup: one wave's LDS accesses complete in order and need no barrier.
__device__ __forceinline__ void group_sync()
{
	if (blockDim.x > 64)
		__syncthreads();
	else
	{
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
	}
}

// Workgroups are dispatched to the 8 XCDs in turn; this order gives each XCD one run of neighbouring tasks, so that
// tasks which share cache lines or DRAM pages run behind one L2.  Measured on in-place passes over 2 GB: contiguous
// rows 5.3 -> 5.6 TB/s, y columns of 128 bytes 4.8 -> 5.1, z columns 4.4 -> 4.9 TB/s.
__device__ __forceinline__ int64_t xcd_order(int64_t b, int64_t W)
{
	const int64_t W8 = W - W % 8;
	return b < W8 ? (b % 8) * (W8 / 8) + b / 8 : b;
}

__device__ __forceinline__ uint32_t fdivu(uint32_t n, uint32_t mul, int shift)
{
	return (uint32_t)(((uint64_t)n * mul) >> shift);
}

using raw16 = uint32_t __attribute__((ext_vector_type(4)));
using raw16u = uint32_t __attribute__((ext_vector_type(4), aligned(2)));

// 4 stored elements at element alignment (rows need not start on a 16-byte boundary)
template <int K>
struct unaligned4
{
	using type = typename store_of<K>::elem __attribute__((ext_vector_type(4), aligned(sizeof(typename store_of<K>::elem))));
};

// The last n = 1, 2 or 3 (uniform) of 4 components, in one store
template <int K>
__device__ __forceinline__ void store_last(typename store_of<K>::elem* p, typename unaligned4<K>::type y, int n)
{
	using elem = typename store_of<K>::elem;
	using e2 = elem __attribute__((ext_vector_type(2), aligned(sizeof(elem))));
	using e3 = elem __attribute__((ext_vector_type(3), aligned(sizeof(elem))));
	if (n == 1)
		gstore(p + 3, (elem)y[3]);
	else if (n == 2)
		gstore((e2*)(p + 2), e2 { y[2], y[3] });
	else
	{
		if constexpr (K == store_f32)
			*(__attribute__((address_space(1))) e3*)(p + 1) = e3 { y[1], y[2], y[3] };
		else
		{
			gstore(p + 1, (elem)y[1]);
			gstore((e2*)(p + 2), e2 { y[2], y[3] });
		}
	}
}

// ---- one lane per (column of 4 consecutive elements, block) --------------------------------------------------------
//
// y, z: a task is C neighbouring columns: C lanes read one contiguous segment, and the 64 / C blocks of a wave the
// segments m planes or rows apart.  Columns are flattened positions (x*S + s along y, (y*X + x)*S + s along z), so 4
// need not divide S: each component takes its own substrate's constants.  Where 4 does not divide the range, its last
// column is moved back to end with the range; it computes all 4 components and stores only those that no other
// column owns.
//
// x, S a multiple of 4: the same with the elements of a voxel for a range.  A lane's loads walk along its row, so a
// cache line is fetched once and hit by the loads that follow.  Rows staged through LDS with coalesced copies instead
// took 24 against 13 us on 100^3 x 4, 89 against 75 us on 200^3 x 8, 890 against 850 us on 400^3 x 8, and in FP16 746
// against 576 us.
//
// BACK: a range that 4 does not divide, with its own kernels, as the stores of parts of a column cost the others
// registers (FP16, 16 elements: 153 -> 196, 400^3 x 8 x sweep 0.56 -> 0.78 ms).
//
// NT: densities that exceed the 256 MB Infinity Cache are streamed past it on y and z.  400^3 x 8, whole diffusion
// solve: FP32 2.96 -> 2.65 ms, FP16 1.90 -> 1.85 ms; along x, whose lines are hit several times, it costs twice the
// time.
template <int M, bool FULL, int K, bool NT, bool BACK>
__device__ __forceinline__ void filter_columns_task(const filter_args& a, int64_t task, float* lt,
													typename vec_of<4>::type* sh, bool first)
{
	using vec = typename vec_of<4>::type;
	using elem = typename store_of<K>::elem;
	using uv = typename unaligned4<K>::type;
	filter_place at;
	const int tid = fresh_lane_value(threadIdx.x);
	at.lane = tid & 63;
	at.wave = tid >> 6;
	at.waves = blockDim.x >> 6;
	at.dist = at.slots = 1 << a.clog;
	at.slot = at.lane & (at.slots - 1);
	at.i = at.lane >> a.clog;
	at.kw = a.kw;
	at.k = at.wave * a.kw + at.i;
	at.last = a.blocks - 1;
	const uint32_t col = (uint32_t)(task << a.clog) + at.slot;
	at.active = col < a.columns && at.k <= at.last;
	const int k = at.active ? at.k : 0;
	const uint32_t cl = at.active ? col : 0;
	const uint32_t outer = fdivu(cl, a.row_mul, a.row_shift);
	const uint32_t q0 = (cl - outer * a.row_columns) * 4;
	// components owned by the column before
	const int back = BACK ? max(0, (int)(q0 + 4 - (uint32_t)a.row_elems)) : 0;
	const uint32_t q = q0 - back;
	const int64_t off = outer * a.outer_stride + q + (int64_t)(k * M) * a.stride;
	const int64_t stride = fresh_uniform(a.stride);
	const int S = fresh_uniform(a.S);
	const int mk = FULL || k < at.last ? M : a.mlast; // (of lanes that read)

	int s[4];
	const uint32_t vox = fdivu(q, a.s_mul, a.s_shift); // voxel of the first component within the row range
	s[0] = (int)(q - vox * (uint32_t)S);
#pragma unroll
	for (int c = 1; c < 4; c++)
		s[c] = s[c - 1] + 1 == S ? 0 : s[c - 1] + 1;

	float t[table_regs];
	if (first)
		table_load<K>(a, t);
	const elem* p = (const elem*)a.data + off;
	constexpr int N = sure<M, FULL>();
	uv raw[M];
	// Lanes past the columns or the line read the first column's first block, elements past a block its first one.
	// Addresses step from element to element behind the compiler's back, here and at the stores: it would hold M
	// multiples of the stride in scalar registers, and spill them, or the loads' M addresses for the stores.
	const elem* pj = p;
#pragma unroll
	for (int j = 0; j < M; j++)
	{
		const uv* src = (const uv*)(j < N || j < mk ? pj : p);
		raw[j] = NT ? __builtin_nontemporal_load(src) : gload(src);
		pj += stride;
		asm volatile("" : "+v"(pj));
	}
	if (first)
	{
		table_store<K>(a, t, lt);
		group_sync();
	}
	auto row = [&](int r) -> vec {
		const float* x = lt + r * S;
		if (S % 4 == 0)
			return *(const vec*)(x + s[0]);
		return vec { x[s[0]], x[s[1]], x[s[2]], x[s[3]] };
	};
	vec v[M];
	const vec gain = row(fr_s);
#pragma unroll
	for (int j = 0; j < M; j++)
	{
		v[j] = __builtin_convertvector(raw[j], vec) * gain;
		if (j >= N)
			v[j] = j < mk ? v[j] : vec(0.f);
	}
	elem* o = (elem*)a.data + off + (mk - 1) * stride;
	asm volatile("" : "+v"(o));
	uint32_t h = K == store_f32 ? 0u : sr_seed(off, rounding_key(a.rounding, 1 + a.axis));
	const int part = fresh_uniform((int)(a.row_elems & 3)); // components that a moved-back column owns
	filter_line<M, FULL, 4>(v, row, mk, a.blocks, at, sh, [&](int j, vec x) {
		uv y;
		if constexpr (K == store_f32)
			y = x;
		else
		{
#pragma unroll
			for (int c = 0; c < 4; c += 2)
			{
				h = xorshift32(h);
				const auto pr = sr_pair<K>(x[c], x[c + 1], h);
				y[c] = pr[0];
				y[c + 1] = pr[1];
			}
		}
		if (!BACK || back == 0)
		{
			if constexpr (NT)
				__builtin_nontemporal_store(y, (uv*)o);
			else
				gstore((uv*)o, y);
		}
		else
			store_last<K>(o, y, part);
		o -= stride;
		asm volatile("" : "+v"(o));
	});

	// Dirichlet faces, written over the solved values in the order x-, x+, y-, y+, z-, z+
	// (host/dirichlet_solver.cpp:91-110): a face of this axis at the line's ends, a face of another axis through the
	// whole line.  Same lane, same addresses: the later store stays.
	if (a.fcond && at.active)
	{
		o += stride; // the block's first element
		const float* ls = lt + a.table_floats;
		auto scale = [&]() { return vec { ls[s[0]], ls[s[1]], ls[s[2]], ls[s[3]] }; };
		for (int d = 0; d < a.dims; d++)
		{
			if (d == a.axis)
			{
#pragma unroll
				for (int mx = 0; mx < 2; mx++)
					if (at.k == (mx ? at.last : 0))
					{
						const vec on = row(mx ? fr_max_on : fr_min_on);
						vec val = row(mx ? fr_max : fr_min);
						if constexpr (K != store_f32)
							val = val * scale();
#pragma unroll
						for (int c = 0; c < 4; c++)
							if (on[c] != 0.f && c >= back)
								gstore(o + (mx ? mk - 1 : 0) * stride + c, (elem)val[c]);
					}
				continue;
			}
#pragma unroll
			for (int c = 0; c < 4; c++)
			{
				if (c < back)
					continue;
				// coordinate d of this component's voxel (its components may lie in different voxels)
				// x: outer = z*Y + y; y: outer = z, vc = x; z: vc = y*X + x
				const uint32_t vc = fdivu(q + c, a.s_mul, a.s_shift);
				const uint32_t hi = fdivu(a.axis == 0 ? outer : vc, a.x_mul, a.x_shift);
				const uint32_t lo = (a.axis == 0 ? outer : vc) - hi * (uint32_t)a.grid[a.axis == 0 ? 1 : 0];
				const int cd = (int)(a.axis == 0 ? (d == 1 ? lo : hi) : a.axis == 1 ? (d == 0 ? vc : outer) : (d == 0 ? lo : hi));
				const int sc = (int)(q + c - vc * (uint32_t)S);
				for (int mx = 0; mx < 2; mx++)
				{
					if (cd != (mx ? a.grid[d] - 1 : 0) || !gload(a.fcond + (2 * d + mx) * S + sc))
						continue;
					float val = gload(a.fval + (2 * d + mx) * S + sc);
					if constexpr (K != store_f32)
						val *= ls[sc];
					for (int j = 0; j < mk; j++)
						gstore(o + j * stride + c, (elem)val);
				}
			}
		}
	}
}

template <int M, bool FULL, int K, bool NT, bool BACK>
__global__ __launch_bounds__(512) void filter_columns_kernel(filter_args a)
{
	extern __shared__ raw16 filter_lds[];
	using vec = typename vec_of<4>::type;
	// two exchange areas in turn: a wave may still read one pass's while another writes the next one's
	const int area = (2 * (blockDim.x >> 6) + 1) << a.clog;
	vec* sh = (vec*)((char*)filter_lds + a.exchange_at);
	int parity = 0;
	bool first = true;
	for (int64_t t = xcd_order(blockIdx.x, gridDim.x); t < a.tasks; t += gridDim.x, parity ^= 1, first = false)
		filter_columns_task<M, FULL, K, NT, BACK>(a, t, (float*)filter_lds, sh + parity * area, first);
}

// ---- x, substrate counts that 4 does not divide: rows staged through LDS, one element per lane and position --------
//
// A workgroup (one wave, or several for long rows) copies whole rows (contiguous in memory) to LDS with
// 16-byte accesses, runs the lines from there and copies the rows back; m is odd, so that the LDS reads of
// neighbouring blocks fall in different banks.  One wave's LDS accesses complete in order and need no barrier.
// The 16-byte pieces of a task's rows that a thread moves (passes == 1: the rows fill at most 64 lanes x M positions
// per wave).  A workgroup loads its next task's rows into registers before it solves the present one.
template <int M, int K>
struct row_pieces
{
	static constexpr int elem_bytes = K == store_f32 ? 4 : 2;
	static constexpr int count = (M * elem_bytes + 15) / 16;
	raw16 piece[count];
	typename store_of<K>::elem tail; // the rows' last elements, fewer than a piece
};

template <int K>
struct row_range
{
	static constexpr int VE = K == store_f32 ? 4 : 8; // elements of a piece
	int64_t row0;
	int nrows, nel, nvec;
	typename store_of<K>::elem* g;
	__device__ __forceinline__ row_range(const filter_args& a, int64_t task)
	{
		row0 = task * a.rows;
		nrows = (int)min((int64_t)a.rows, a.total_rows - row0);
		nel = nrows * (int)a.row_elems;
		nvec = nel / VE;
		g = (typename store_of<K>::elem*)a.data + row0 * a.row_elems;
	}
};

template <int M, int K>
__device__ __forceinline__ void rows_fetch(const filter_args& a, int64_t task, row_pieces<M, K>& x)
{
	const row_range<K> r(a, task);
	const int tid = fresh_lane_value(threadIdx.x), nthr = blockDim.x;
#pragma unroll
	for (int j = 0; j < row_pieces<M, K>::count; j++)
		x.piece[j] = gload((const raw16u*)r.g + min(tid + nthr * j, r.nvec - 1)); // past the end: the last one again
	x.tail = gload(r.g + min(r.nvec * r.VE + tid, r.nel - 1));
}

template <int M, int K>
__device__ __forceinline__ void rows_put(const filter_args& a, int64_t task, const row_pieces<M, K>& x, char* rows)
{
	const row_range<K> r(a, task);
	const int tid = fresh_lane_value(threadIdx.x), nthr = blockDim.x;
#pragma unroll
	for (int j = 0; j < row_pieces<M, K>::count; j++)
		((raw16*)rows)[min(tid + nthr * j, r.nvec - 1)] = x.piece[j];
	// rows longer than the pieces (several passes)
	for (int i = tid + nthr * row_pieces<M, K>::count; i < r.nvec; i += nthr)
		((raw16*)rows)[i] = gload((const raw16u*)r.g + i);
	if (tid < r.nel - r.nvec * r.VE)
		((typename store_of<K>::elem*)rows)[r.nvec * r.VE + tid] = x.tail;
}

// The staged rows of one task: solve, Dirichlet faces, copy back.
template <int M, bool FULL, int K>
__device__ __forceinline__ void filter_rows_task(const filter_args& a, int64_t task, char* lds)
{
	using elem = typename store_of<K>::elem;
	const int tid = fresh_lane_value(threadIdx.x), nthr = blockDim.x;
	const int S = fresh_uniform(a.S), XS = (int)a.row_elems;
	const row_range<K> rg(a, task);
	const int64_t row0 = rg.row0;
	const int nrows = rg.nrows, nvec = rg.nvec;
	elem* g = rg.g;
	elem* l = (elem*)(lds + a.rows_at);
	const float* lt = (const float*)lds;
	const float* ls = lt + a.table_floats;

	filter_place at;
	at.lane = tid & 63;
	const bool whole = a.kw == a.blocks; // each wave has whole lines
	const int wave = tid >> 6, waves = nthr >> 6;
	at.wave = whole ? 0 : wave;
	at.waves = whole ? 1 : waves;
	at.dist = at.slots = a.lines_pass;
	at.slot = at.lane % a.lines_pass;
	const int b = at.lane / a.lines_pass;
	at.kw = a.kw;
	at.i = b % a.kw;
	at.k = at.wave * a.kw + at.i;
	at.last = a.blocks - 1;
	const int mk = FULL || at.k < at.last ? M : a.mlast;
	constexpr int N = sure<M, FULL>();

	for (int pass = 0; pass < a.passes; pass++)
	{
		if (pass > 0 && at.waves > 1)
			__syncthreads(); // the exchange area of the pass before
		const int first = (whole ? pass * waves + wave : pass) * a.lines_pass + at.slot;
		const int r = (int)fdivu((uint32_t)first, a.s_mul, a.s_shift), line = first - r * S;
		at.active = b < a.kw && at.k <= at.last && r < nrows;
		const int pos = r * XS + at.k * M * S + line;
		float v[M];
		auto row = [&](int rw) { return lt[rw * S + line]; };
		const float gain = row(fr_s);
		const elem* lv = l + (at.active ? pos : 0); // inactive lanes read what is there
#pragma unroll
		for (int j = 0; j < M; j++)
		{
			v[j] = (float)lv[j < N || j < mk ? j * S : 0] * gain;
			if (j >= N)
				v[j] = j < mk ? v[j] : 0.f;
		}
		uint32_t h = K == store_f32 ? 0u : sr_seed(row0 * XS + pos, rounding_key(a.rounding, 1));
		const int So = fresh_uniform(S); // the stores' addresses are not the loads' held
		elem* lo = l + pos;
		filter_line<M, FULL, 1>(v, row, mk, a.blocks, at, (float*)(lds + a.exchange_at), [&](int j, float x) {
			elem* o = lo + j * So;
			if constexpr (K == store_f32)
				*o = x;
			else
			{
				h = xorshift32(h);
				*o = sr_pair<K>(x, 0.f, h)[0];
			}
		});
		// Dirichlet x faces at the row's ends
		if (a.fcond && at.active)
			for (int mx = 0; mx < 2; mx++)
				if (at.k == (mx ? at.last : 0) && row(mx ? fr_max_on : fr_min_on) != 0.f)
				{
					const float val = row(mx ? fr_max : fr_min);
					l[pos + (mx ? mk - 1 : 0) * S] = (elem)(K == store_f32 ? val : val * ls[line]);
				}
	}
	group_sync();
	// then the rows on y and z faces, in the order y-, y+, z-, z+ (host/dirichlet_solver.cpp:91-110)
	if (a.fcond)
	{
		bool any = false;
		for (int rr = 0; rr < nrows; rr++)
		{
			const uint32_t row = (uint32_t)(row0 + rr), z = fdivu(row, a.row_mul, a.row_shift);
			const int y = (int)(row - z * (uint32_t)a.grid[1]);
			for (int f = 2; f < 2 * a.dims; f++)
			{
				if ((f < 4 ? y : (int)z) != ((f & 1) ? a.grid[f >> 1] - 1 : 0))
					continue;
				any = true;
				for (int i = tid; i < XS; i += nthr)
				{
					const int sc = i % S;
					if (!gload(a.fcond + f * S + sc))
						continue;
					float val = gload(a.fval + f * S + sc);
					if constexpr (K != store_f32)
						val *= ls[sc];
					l[rr * XS + i] = (elem)val;
				}
			}
		}
		if (any)
			group_sync();
	}
	constexpr int U = row_pieces<M, K>::count;
	raw16 w[U];
#pragma unroll
	for (int j = 0; j < U; j++)
		w[j] = ((const raw16*)l)[min(tid + nthr * j, nvec - 1)];
#pragma unroll
	for (int j = 0; j < U; j++)
		gstore((raw16u*)g + min(tid + nthr * j, nvec - 1), (raw16u)w[j]);
	for (int i = tid + nthr * U; i < nvec; i += nthr)
		gstore((raw16u*)g + i, (raw16u)((const raw16*)l)[i]);
	if (tid < rg.nel - nvec * rg.VE)
		gstore(g + nvec * rg.VE + tid, l[nvec * rg.VE + tid]);
}

template <int M, bool FULL, int K>
__global__ __launch_bounds__(512) void filter_rows_kernel(filter_args a)
{
	extern __shared__ raw16 filter_lds[];
	char* lds = (char*)filter_lds;
	row_pieces<M, K> x;
	float tab[table_regs];
	int64_t t = xcd_order(blockIdx.x, gridDim.x);
	table_load<K>(a, tab);
	rows_fetch<M, K>(a, t, x);
	table_store<K>(a, tab, (float*)lds);
	for (; t < a.tasks; t += gridDim.x)
	{
		rows_put<M, K>(a, t, x, lds + a.rows_at);
		group_sync();
		if (t + gridDim.x < a.tasks)
			rows_fetch<M, K>(a, t + gridDim.x, x);
		filter_rows_task<M, FULL, K>(a, t, lds);
		group_sync(); // the next rows are staged over these
	}
}

// ---- many small meshes in one launch --------------------------------------------------------------------------------
//
// A small mesh (small_filter) is bound by its launches and their latency; the small instances of a batch share one launch
// per axis.  A workgroup (one wave) finds its instance among the running task counts and the
// block length by a branch; the arguments are read from memory.
template <int K, int... Ms>
__device__ __forceinline__ void small_columns(const filter_args& a, int64_t task, raw16* lds)
{
	auto* sh = (typename vec_of<4>::type*)((char*)lds + a.exchange_at);
	((a.m == Ms ? filter_columns_task<Ms, false, K, false, true>(a, task, (float*)lds, sh, true) : void()), ...);
}
template <int M, int K>
__device__ __forceinline__ void small_rows_of(const filter_args& a, int64_t task, raw16* lds)
{
	row_pieces<M, K> x;
	float tab[table_regs];
	table_load<K>(a, tab);
	rows_fetch<M, K>(a, task, x);
	table_store<K>(a, tab, (float*)lds);
	rows_put<M, K>(a, task, x, (char*)lds + a.rows_at);
	group_sync();
	filter_rows_task<M, false, K>(a, task, (char*)lds);
}
template <int K, int... Ms>
__device__ __forceinline__ void small_rows(const filter_args& a, int64_t task, raw16* lds)
{
	((a.m == Ms ? small_rows_of<Ms, K>(a, task, lds) : void()), ...);
}

template <int K>
__global__ __launch_bounds__(64) void filter_small_kernel(const filter_args* __restrict__ inst,
														  const int* __restrict__ first, int count)
{
	extern __shared__ raw16 filter_lds[];
	const int b = (int)xcd_order(blockIdx.x, gridDim.x);
	int lo = 0, hi = count - 1; // first[lo] <= b < first[hi + 1]
	while (lo < hi)
	{
		const int mid = (lo + hi + 1) / 2;
		if (first[mid] <= b)
			lo = mid;
		else
			hi = mid - 1;
	}
	const int i = __builtin_amdgcn_readfirstlane(lo);
	const filter_args& a = inst[i];
	const int64_t task = b - first[i];
	if (a.staged)
		small_rows<K, 3, 5, 7, 9, 11, 13, 15, 17>(a, task, filter_lds);
	else
		small_columns<K, 2, 3, 4, 5, 7, 9, 11, 13, 14, 16>(a, task, filter_lds);
}

// ---- host side ------------------------------------------------------------------------------------------------------


// block lengths the kernels are built for: odd ones where the rows are staged (LDS banks)
static constexpr int column_blocks[] = { 2, 3, 4, 5, 7, 9, 11, 13, 14, 16, 18, 20, 22, 25 };
static constexpr int row_blocks[] = { 3, 5, 7, 9, 11, 13, 15, 17, 19, 21, 23, 25 };

// f(block length, every block full) as compile-time constants, for the lengths listed
template <int... Ms, typename F>
static void by_block(int m, bool full, F&& f)
{
	auto one = [&](auto c) {
		if (c == m)
			full ? f(c, std::true_type()) : f(c, std::false_type());
	};
	(one(std::integral_constant<int, Ms>()), ...);
}

// The filter needs 0 <= mu < 1, i.e. a >= 0 and 1 + decay*dt/dims > 0, and it is used up to mu = 0.73 (a = 10), where its
// FP32 error against FP64 solves is still no larger than the partitioned sweep's.  Worst of 144 lines of 100, 400 and
// 1000 voxels each (filter / partitioned), point source, relative L2 and per voxel above 1e-3 of the largest:
//   a = 1..2.5    1.1e-7 / 1.3e-7  6.7e-7 / 7.0e-7        a = 16..25     1.8e-7 / 2.6e-7  1.3e-6 / 7.8e-7
//   a = 6..10     1.7e-7 / 2.5e-7  8.6e-7 / 9.7e-7        a = 100..300   4.0e-7 / 3.7e-7  3.3e-6 / 7.1e-7
//   a = 10..16    1.7e-7 / 2.5e-7  1.1e-6 / 8.8e-7        a = 1e3..1e5   3.2e-6 / 4.6e-7  1.7e-5 / 8.1e-7
// (uniform random densities hide it: 2.0e-7 / 3.2e-7 at a = 1e3..1e5).
static constexpr double filter_largest_mu = 0.73;
static bool filter_coefficients_ok(const bfvm_ctx* ctx, int axis)
{
	const double h2 = (double)ctx->mesh.vs[axis] * ctx->mesh.vs[axis];
	for (int s = 0; s < ctx->mesh.S; s++)
	{
		const double a = (double)ctx->mesh.dt * ctx->D[s] / h2;
		const double lam = 1.0 + (double)ctx->decay[s] * ctx->mesh.dt / ctx->mesh.dims;
		if (!(a >= 0.0) || !(lam > 0.0) || !std::isfinite(a) || !std::isfinite(lam))
			return false;
		if (!(2.0 * a / (lam + 2.0 * a + std::sqrt(lam * (lam + 4.0 * a))) <= filter_largest_mu))
			return false;
	}
	return true;
}

// Workgroups: enough that every SIMD holds two waves, while blocks stay long (fewer exchanges, wider loads).
static constexpr int64_t filter_fill_waves = 2048;
static constexpr int filter_max_waves = 8; // waves of a workgroup
static constexpr int64_t infinity_cache_bytes = (int64_t)256 << 20;

// LDS bytes of the coefficient table and the storage scales, to the next vector
static int filter_lds_table(const bfvm_ctx* ctx, int blocks, int kw)
{
	const int S = ctx->mesh.S;
	const int64_t floats = (int64_t)(fr_ends + 2 * blocks + kw) * S + (ctx->storage == BFVM_STORAGE_F32 ? 0 : S);
	return (int)std::min<int64_t>((floats * 4 + 15) / 16 * 16, 1 << 20);
}

// Expected time of an element, up to a factor: a block's scan costs about 8 elements; lanes without elements (the share
// `used` has them) hold no loads in flight; blocks of at most 16 elements leave room for 3 waves per SIMD, longer ones
// for 2; a short last block takes selects; more than 4 waves per workgroup wait for each other.  Measured (ms, y / z,
// FP32 c3 = 8 columns, 16-bit c4 = 16 columns): 400^3 x 8 FP32 16 elements 0.68 / 0.71, 25 elements 0.73 / 0.76, 9
// elements 0.87 / 0.88; FP16 25 elements 0.46 / 0.49, 16 elements (7 waves) 0.78 / 0.78; 256^3 x 16 BF16 16 elements
// 0.26 / 0.30, 22 elements (short last block, 3 waves) 0.34 / 0.37; 200^3 x 8 FP32 25 elements 0.068 / 0.071, 16
// elements 0.069 / 0.072; 100^3 x 4 FP32 13 elements (8 blocks) 0.012 / 0.011, 25 (4 blocks) 0.013 / 0.012.
static double filter_cost(int m, int waves, bool full, double used)
{
	return (m + 8.0) / m * std::pow(used, -0.4) * (m <= 16 ? 0.75 : 1.0) * (full ? 1.0 : 1.15) * (waves > 4 ? 1.5 : 1.0);
}

// Staged rows: lanes without a line cost their full share, and larger workgroups wait for each other.
static double row_waves_factor(int waves) { return waves > 4 ? 0.75 : waves > 2 ? 0.95 : 1.0; }
static double row_cost(const filter_plan& p, bool full, double used)
{
	return (p.m + 8.0) / p.m / used * (full ? 1.0 : 1.05) / row_waves_factor(p.waves);
}

// `shared`: for a launch shared with other instances (filter_small_kernel): one wave per workgroup that holds whole lines,
// and the block lengths that kernel is built for.
filter_plan choose_filter(const bfvm_ctx* ctx, int axis, bool shared)
{
	const int most_waves = shared ? 1 : filter_max_waves;
	// rows of a task in LDS: one wave with 24 KB leaves a CU six waves (shared launches of 20 instances of 32..64 voxels an
	// edge, FP32 with gradients 254 us, with 8 KB 229)
	const int64_t most_row_bytes = shared ? 8 * 1024 : 24 * 1024;
	const auto& g = ctx->mesh;
	const int n = g.grid[axis], S = g.S;
	const int64_t XS = (int64_t)g.grid[0] * S, e = (int64_t)storage_bytes(ctx->storage);
	filter_plan best, quick;
	double best_cost = 0, quick_cost = 0;
	if (n < 2 || !filter_coefficients_ok(ctx, axis))
		return best;
	// best: the cheapest lengths; quick: the shortest chain of operations, for meshes that do not fill the card anyway
	auto consider = [&](const filter_plan& p, double used) {
		const int waves = p.kw < p.blocks ? p.waves : 1; // that a line takes
		const double cost = p.staged && waves == 1 ? row_cost(p, n % p.m == 0, used)
												   : filter_cost(p.m, waves, n % p.m == 0, used);
		const double chain = std::max(p.m, 7) + 8 * waves;
		if (best.blocks == 0 || cost < best_cost)
		{
			best = p;
			best_cost = cost;
		}
		if (quick.blocks == 0 || chain < quick_cost)
		{
			quick = p;
			quick_cost = chain;
		}
	};
	// a line's last block holds at least half its length (sure)
	auto fits = [&](int m) { return n - ((n + m - 1) / m - 1) * m >= m / 2; };
	// x rows of a substrate count that 4 does not divide go through LDS where a row fits there; direct columns of 4
	// overlap, and their last one stores in parts.  Staged / direct, us: 160^3 x 5 FP32 25 / 58, FP16 28 / 62; 160^3 x 7
	// 35 / 62, 36 / 79; 160^3 x 13 54 / 77, 67 / 73; 134x200x143 x 15 60 / 79, 75 / 90; 400x200x200 x 7 159 / 310, 111 /
	// 260; 256^3 x 5 122 / 278, 118 / 207; 147x127x200 x 14 57 / 71, but FP16 71 / 63.
	const int64_t rows = (int64_t)g.grid[1] * g.grid[2];
	if (axis == 0 && S % 4 != 0 && XS * e >= 16 && rows < (int64_t)1 << 31)
	{
		const int L = S;
		for (int m : row_blocks)
		{
			if (!fits(m) || (shared && (m > 17 || (n + m - 1) / m > 64)))
				continue;
			filter_plan p;
			p.m = m;
			p.blocks = (n + m - 1) / m;
			p.staged = true;
			if (p.blocks <= 64)
			{
				// whole lines in each wave, of as many rows as fill the waves best
				p.lines_pass = 64 / p.blocks;
				p.kw = p.blocks;
				double best_used = 0;
				for (int r = 1; r <= 16 && (r == 1 || r * XS * e <= most_row_bytes); r++)
				{
					const int groups = (r * L + p.lines_pass - 1) / p.lines_pass, waves = std::min(groups, most_waves);
					const int passes = (groups + waves - 1) / waves;
					const double used = (double)r * L / (waves * passes * p.lines_pass) * row_waves_factor(waves);
					if (used > best_used * 1.02)
					{
						best_used = used;
						p.rows = r;
						p.waves = waves;
						p.passes = passes;
					}
				}
			}
			else
			{
				// one row: as many of its lines side by side as a wave holds, their blocks over several waves
				p.lines_pass = std::min({ L, 64, std::max(1, 64 * filter_max_waves / p.blocks) });
				p.kw = std::min(64 / p.lines_pass, p.blocks);
				p.waves = (p.blocks + p.kw - 1) / p.kw;
				p.rows = 1;
				p.passes = (L + p.lines_pass - 1) / p.lines_pass;
			}
			if (p.waves > most_waves)
				continue;
			p.exchange_at = filter_lds_table(ctx, p.blocks, p.kw);
			p.rows_at =
				p.exchange_at + (p.kw < p.blocks ? ((2 * p.waves + 1) * p.lines_pass * 4 + 15) / 16 * 16 : 0);
			const int64_t lds = p.rows_at + (p.rows * XS * e + 15) / 16 * 16;
			if (lds > 64 * 1024)
				continue;
			p.lds = (int)lds;
			p.tasks = (rows + p.rows - 1) / p.rows;
			p.lines_group = p.rows * L;
			consider(p, (double)p.rows * L * n / (64.0 * p.waves * m * p.passes));
		}
	}
	if (best.blocks == 0)
	{
		const int64_t row_elems = axis == 0 ? S : axis == 1 ? XS : (int64_t)g.grid[1] * XS;
		const int64_t row_columns = (row_elems + 3) / 4;
		const int64_t columns = row_columns * (axis == 0 ? (int64_t)g.grid[1] * g.grid[2] : axis == 1 ? g.grid[2] : 1);
		if (row_elems < 4 || columns >= ((int64_t)1 << 31) / 4)
			return best;
		// y, z: 128-byte segments (8 lanes of FP32, 16 of 16-bit storage): a wave whose segments are 64 bytes reaches
		// 4.2-4.7 TB/s on 2 GB, with 128 bytes 4.8-5.2 TB/s.  x: 4 rows side by side (400^3 x 8 FP16 0.58 ms, one row 0.65,
		// 256^3 x 16 BF16 0.25, one row 0.33 ms).  Long lines take fewer columns where 8 waves cannot hold them.
		int widest = e == 4 ? 3 : 4;
		if (axis == 0)
			for (widest = 2; widest < 5 && (1 << widest) < S; widest++)
				;
		for (int clog = widest; clog >= 0 && best.blocks == 0; clog--)
			for (int m : column_blocks)
			{
				if (!fits(m) || (shared && m > 16))
					continue;
				filter_plan p;
				p.m = m;
				p.blocks = (n + m - 1) / m;
				p.clog = clog;
				p.kw = 64 >> clog;
				p.waves = (p.blocks + p.kw - 1) / p.kw;
				if (p.waves > most_waves)
					continue;
				p.exchange_at = filter_lds_table(ctx, p.blocks, p.kw);
				p.lds = p.exchange_at + (p.waves > 1 ? 2 * ((2 * p.waves + 1) << clog) * 16 : 0);
				if (p.lds > 64 * 1024)
					continue;
				p.tasks = (columns + (1 << clog) - 1) >> clog;
				p.lines_group = (1 << clog) * (S % 4 == 0 ? 1 : 4);
				consider(p, (double)n / (m * p.kw * p.waves));
			}
	}
	// an instance of a shared launch does not have to fill the card by itself: 20 instances of 32..64 voxels an edge, FP16,
	// 149 us with the short chains, 105 with the cheapest lengths
	filter_plan& p = !shared && best.tasks * best.waves < filter_fill_waves ? quick : best;
	p.streamed = axis != 0 && (int64_t)(ctx->mesh.V * S) * e > infinity_cache_bytes;
	return p;
}

size_t filter_table_floats(const filter_plan& p, int S) { return (size_t)(fr_ends + 2 * p.blocks + p.kw) * S; }

void launch_filter_coefficients(const bfvm_ctx* ctx, int axis, const filter_plan& p, float* tab, hipStream_t stream)
{
	const int S = ctx->mesh.S;
	hipLaunchKernelGGL(filter_coefficients_kernel, dim3((S + 63) / 64), dim3(64), 0, stream, tab, ctx->d_D,
					   ctx->d_decay, ctx->face_val + 2 * axis * S, ctx->face_cond + 2 * axis * S, ctx->mesh.dt,
					   ctx->mesh.vs[axis], ctx->mesh.dims, ctx->mesh.grid[axis], S, p.m, p.blocks, p.kw);
	BFVM_HIP(hipGetLastError());
}

static filter_args make_filter_args(const bfvm_ctx* ctx, int axis, const filter_plan& p, const float* tab)
{
	const auto& g = ctx->mesh;
	filter_args a {};
	a.data = ctx->dens;
	a.scale = ctx->dscale;
	a.rounding = ctx->rounding_step;
	a.fval = ctx->has_faces ? ctx->face_val : nullptr;
	a.fcond = ctx->has_faces ? ctx->face_cond : nullptr;
	a.tab = tab;
	for (int d = 0; d < 3; d++)
		a.grid[d] = g.grid[d];
	a.S = g.S;
	a.dims = g.dims;
	a.axis = axis;
	a.m = p.m;
	a.blocks = p.blocks;
	a.kw = p.kw;
	a.mlast = g.grid[axis] - (p.blocks - 1) * p.m;
	a.tasks = p.tasks;
	a.table_floats = (int)filter_table_floats(p, g.S);
	a.exchange_at = p.exchange_at;
	const int64_t XS = (int64_t)g.grid[0] * g.S;
	fast_divisor((uint32_t)g.S, a.s_mul, a.s_shift);
	fast_divisor((uint32_t)g.grid[axis == 0 ? 1 : 0], a.x_mul, a.x_shift);
	a.staged = p.staged ? 1 : 0;
	if (p.staged)
	{
		a.row_elems = XS;
		a.rows = p.rows;
		a.lines_pass = p.lines_pass;
		a.passes = p.passes;
		a.total_rows = (int64_t)g.grid[1] * g.grid[2];
		a.rows_at = p.rows_at;
		fast_divisor((uint32_t)g.grid[1], a.row_mul, a.row_shift);
		return a;
	}
	const int64_t plane = (int64_t)g.grid[1] * XS;
	a.clog = p.clog;
	a.stride = axis == 0 ? g.S : axis == 1 ? XS : plane;
	a.row_elems = a.stride;
	a.outer_stride = axis == 0 ? XS : axis == 1 ? plane : 0;
	a.row_columns = (uint32_t)((a.row_elems + 3) / 4);
	a.columns = a.row_columns * (uint32_t)(axis == 0 ? (int64_t)g.grid[1] * g.grid[2] : axis == 1 ? g.grid[2] : 1);
	fast_divisor(a.row_columns, a.row_mul, a.row_shift);
	return a;
}

void launch_filter_sweep(bfvm_ctx* ctx, int axis)
{
	const axis_tables& t = ctx->axes[axis];
	const filter_plan& p = t.filter;
	const filter_args a = make_filter_args(ctx, axis, p, t.filter_tab);
	// one task per workgroup unless the caller or the autotuner set a cap: fewer workgroups that fetch their next rows
	// early took 37 against 35 us on 160^3 x 7, 77 against 60 on 134x200x143 x 15 (16 waves per CU)
	const int64_t cap = ctx->sweep_workgroups[axis] > 0 ? ctx->sweep_workgroups[axis] : (int64_t)1 << 24;
	const dim3 blocks((unsigned)std::min(p.tasks, cap)), threads(64 * p.waves);
	const size_t lds = p.lds;
	const bool full = a.mlast == a.m, back = a.row_elems % 4 != 0;
	by_storage(ctx->storage, [&](auto kind) {
		constexpr int K = decltype(kind)::value;
		if (p.staged)
			by_block<3, 5, 7, 9, 11, 13, 15, 17, 19, 21, 23, 25>(p.m, full, [&](auto m, auto f) {
				hipLaunchKernelGGL((filter_rows_kernel<m, f, K>), blocks, threads, lds, ctx->stream, a);
			});
		else
			by_block<2, 3, 4, 5, 7, 9, 11, 13, 14, 16, 18, 20, 22, 25>(p.m, full && !back, [&](auto m, auto f) {
				auto kernel = p.streamed ? filter_columns_kernel<m, f, K, true, false> : filter_columns_kernel<m, f, K, false, false>;
				if constexpr (!f)
					if (back)
						kernel = p.streamed ? filter_columns_kernel<m, f, K, true, true> : filter_columns_kernel<m, f, K, false, true>;
				hipLaunchKernelGGL(kernel, blocks, threads, lds, ctx->stream, a);
			});
	});
	BFVM_HIP(hipGetLastError());
}

// Whether an instance of a batch takes its sweeps in the launches shared by the small ones: every axis has a plan for
// them, and its densities are at most 8 MB, where a launch of its own is bound by latency and the steps between
// launches.  us per step at 4 / 8 / 16 / 32 MB, edges from 32: 20 instances up to 64, FP16 130 / 118 / 119 / 120, FP32
// with gradients 270 / 250 / 264 / 265; 10 up to 96, FP16 161 / 138 / 154 / 158, FP32 314 / 267 / 270 / 289; 12 up to
// 120, FP16 196 / 202 / 221 / 219, FP32 420 / 370 / 381 / 468; 19 up to 200, FP16 1080 / 1055 / 1084 / 1177.  All in
// launches of their own: 166 and 268 for the first two, and with one-launch batches before the filter 199 and 346.
bool small_filter(const bfvm_ctx* ctx)
{
	if ((int64_t)(ctx->mesh.V * ctx->mesh.S) * (int64_t)storage_bytes(ctx->storage) > (int64_t)8 << 20)
		return false;
	for (int axis = 0; axis < ctx->mesh.dims; axis++)
		if (choose_filter(ctx, axis, true).blocks == 0)
			return false;
	return true;
}

size_t small_filter_args_bytes() { return sizeof(filter_args); }
void small_filter_args(const bfvm_ctx* ctx, int axis, void* out, int& tasks, int& lds)
{
	const filter_plan& p = ctx->axes[axis].filter;
	*(filter_args*)out = make_filter_args(ctx, axis, p, ctx->axes[axis].filter_tab);
	tasks = (int)p.tasks;
	lds = p.lds;
}

void launch_small_filters(int storage, hipStream_t stream, const void* inst, const int* first, int count, int tasks, int lds)
{
	by_storage(storage, [&](auto kind) {
		hipLaunchKernelGGL(filter_small_kernel<decltype(kind)::value>, dim3((unsigned)tasks), dim3(64), (size_t)lds,
						   stream, (const filter_args*)inst, first, count);
	});
	BFVM_HIP(hipGetLastError());
}

} // namespace bfvm
