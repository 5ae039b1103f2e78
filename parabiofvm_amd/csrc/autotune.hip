// Launch-shape autotuner.  The reference fixes its device launch shapes (work_block_size = 30 in
// CUDA/diffusion_solver.cpp:11, 256-thread blocks in CUDA/diffusion_solver.cu:947-987); here the shapes of
// every sweep axis (register chunk, lines per workgroup, workgroup count) and of the gradient (workgroups it
// aims for) are picked by timing candidates on the context's own mesh, and cached per (axis, mesh shape,
// substrate count, storage, whether the axis takes the recursive filter) for the process, so that contexts of the same
// shape tune once.  A batch's
// instances keep their own shapes.  The cache can be written to and read
// from a text file, so that a later process starts tuned.
#include <array>
#include <cstdio>
#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <tuple>

#include "bfvm_internal.hpp"

namespace bfvm {

namespace {

struct sweep_shape
{
	int chunk = 0, lines = 0, workgroups = 0;
	// a shape of the recursive filter (its entries hold a workgroup cap only), or one of the partitioned sweep
	bool filter() const { return chunk == 0 && lines == 0; }
};

// axis (or -1: gradient), X, Y, Z, S, storage, algorithm, recursive filter.  Whether an axis takes the filter depends on
// the coefficients too, and neither sweep's shape serves the other: a chunk asks for the partitioned sweep.
using shape_key = std::tuple<int, int, int, int, int, int, int, bool>;

std::mutex g_cache_mutex;
std::map<shape_key, sweep_shape> g_sweep_cache;
struct gradient_shape
{
	int groups = 0;
	bool stacked = false;
	int order = 0;
};
std::map<shape_key, gradient_shape> g_gradient_cache;
// "gradient" lines of files from before the branch-free gradient: they shaped its tiles, and would now put its marching
// form where the automatic one is up to 2.6 times faster; read and written back, not used
std::map<shape_key, gradient_shape> g_tile_gradients;
// "batch" lines, from when batches had launch shapes of their own: read and written back, not used
std::map<std::string, std::array<int, 18>> g_batch_lines;

shape_key key_of(const bfvm_ctx* ctx, int axis, bool filter)
{
	const auto& m = ctx->mesh;
	return shape_key { axis, m.grid[0], m.grid[1], m.grid[2], m.S, ctx->storage, ctx->algorithm, filter };
}

// Fastest of `reps` launches after one untimed launch, each timed alone with HIP events on `stream`.
template <typename F>
float best_ms(hipStream_t stream, int reps, F&& launch)
{
	launch();
	hipEvent_t start = nullptr, stop = nullptr;
	BFVM_HIP(hipEventCreate(&start));
	hipError_t err = hipEventCreate(&stop);
	if (err != hipSuccess)
	{
		(void)hipEventDestroy(start);
		BFVM_HIP(err);
	}
	float best = 1e30f;
	try
	{
		for (int r = 0; r < reps; r++)
		{
			BFVM_HIP(hipEventRecord(start, stream));
			launch();
			BFVM_HIP(hipEventRecord(stop, stream));
			BFVM_HIP(hipEventSynchronize(stop));
			float ms = 0;
			BFVM_HIP(hipEventElapsedTime(&ms, start, stop));
			best = std::min(best, ms);
		}
	}
	catch (...)
	{
		(void)hipEventDestroy(start);
		(void)hipEventDestroy(stop);
		throw;
	}
	BFVM_HIP(hipEventDestroy(start));
	BFVM_HIP(hipEventDestroy(stop));
	return best;
}

void apply_sweep_shape(bfvm_ctx* ctx, int axis, const sweep_shape& s)
{
	ctx->chunk_request[axis] = s.chunk;
	ctx->lines_request[axis] = s.lines;
	ctx->sweep_workgroups[axis] = s.workgroups;
	build_partition(ctx, axis, s.chunk, s.lines);
	launch_partition_coefficients(ctx, axis);
}

// Candidates: the automatic shape, or, where that is not the recursive filter, register chunks (16-element blocks
// hold 4-substrate vectors; 16-bit storage instantiates 16 and 32 only) and lines (y, z) or rows (x) per workgroup;
// then the workgroup count of the best of those.  The partitioned shapes are not timed against the filter: on 400^3 x
// 8 their best ran 1.01 / 0.83 / 0.90 ms (x/y/z, FP32) and 0.89 / 0.87 / 0.86 ms (FP16) where the filter takes 0.82 /
// 0.79 / 0.85 and 0.55 / 0.49 / 0.52 ms, and on small meshes it is 2-5 times faster.
sweep_shape search_sweep(bfvm_ctx* ctx, int axis, bool filter, int reps)
{
	std::vector<int> chunks = { 16, 32 };
	if (ctx->storage == BFVM_STORAGE_F32)
		chunks.push_back(64);
	std::vector<int> lines = axis == 0 ? std::vector<int> { 0, 1, 2, 4, 8 } : std::vector<int> { 0, 4, 8, 16, 24, 32 };
	if (filter)
	{
		chunks = { 0 };
		lines = { 0 };
	}
	sweep_shape best;
	float best_t = 1e30f;
	for (int c : chunks)
		for (int l : lines)
		{
			const sweep_shape cand { c, l, 0 };
			try
			{
				apply_sweep_shape(ctx, axis, cand);
			}
			catch (const std::runtime_error&)
			{
				continue; // does not fit the register or LDS budget
			}
			const float t = best_ms(ctx->stream, reps, [&] { launch_sweep(ctx, axis); });
			if (t < best_t)
			{
				best_t = t;
				best = cand;
			}
		}
	if (best_t >= 1e30f)
		throw std::runtime_error("autotune: no sweep shape fits axis " + std::to_string(axis));
	for (int w : { 1024, 2048, 4096, 16384, 65536 })
	{
		sweep_shape cand = best;
		cand.workgroups = w;
		apply_sweep_shape(ctx, axis, cand);
		const float t = best_ms(ctx->stream, reps, [&] { launch_sweep(ctx, axis); });
		if (t < best_t * 0.99f)
		{
			best_t = t;
			best = cand;
		}
	}
	return best;
}

} // namespace

// Text file, one entry per line:
//   sweep <axis> <X> <Y> <Z> <S> <storage> <algorithm> <chunk> <lines> <workgroups>
//     (chunk and lines 0: a shape of the recursive filter, for axes that take it; else one of the partitioned sweep, for
//     axes that do not)
//   gradient_field <X> <Y> <Z> <S> <storage> <algorithm> <workgroups> <stacked> <order>
//   gradient <X> <Y> <Z> <S> <storage> <algorithm> <workgroups> <stacked> [<order>], kept but not used
//   batch <key> <18 numbers>, kept but not used
void save_tuning(const char* path)
{
	std::lock_guard<std::mutex> lock(g_cache_mutex);
	FILE* f = std::fopen(path, "w");
	if (!f)
		throw std::invalid_argument(std::string("cannot write ") + path);
	for (const auto& [k, v] : g_sweep_cache)
		std::fprintf(f, "sweep %d %d %d %d %d %d %d %d %d %d\n", std::get<0>(k), std::get<1>(k), std::get<2>(k),
					 std::get<3>(k), std::get<4>(k), std::get<5>(k), std::get<6>(k), v.chunk, v.lines, v.workgroups);
	for (const auto& [name, cache] : { std::pair { "gradient", &g_tile_gradients }, { "gradient_field", &g_gradient_cache } })
		for (const auto& [k, v] : *cache)
			std::fprintf(f, "%s %d %d %d %d %d %d %d %d %d\n", name, std::get<1>(k), std::get<2>(k), std::get<3>(k),
						 std::get<4>(k), std::get<5>(k), std::get<6>(k), v.groups, v.stacked ? 1 : 0, v.order);
	for (const auto& [k, fields] : g_batch_lines)
	{
		std::fprintf(f, "batch %s", k.c_str());
		for (int v : fields)
			std::fprintf(f, " %d", v);
		std::fprintf(f, "\n");
	}
	const bool bad = std::ferror(f) != 0;
	std::fclose(f);
	if (bad)
		throw std::runtime_error(std::string("error writing ") + path);
}

void load_tuning(const char* path)
{
	FILE* f = std::fopen(path, "r");
	if (!f)
		throw std::invalid_argument(std::string("cannot read ") + path);
	std::string text;
	char buf[4096];
	size_t got;
	while ((got = std::fread(buf, 1, sizeof buf, f)) > 0)
		text.append(buf, got);
	std::fclose(f);
	std::istringstream lines(text);
	std::string line;
	std::lock_guard<std::mutex> lock(g_cache_mutex);
	int lineno = 0;
	while (std::getline(lines, line))
	{
		lineno++;
		if (line.empty())
			continue;
		std::istringstream in(line);
		std::string kind;
		in >> kind;
		bool ok = false;
		if (kind == "sweep")
		{
			int axis, X, Y, Z, S, st, alg;
			sweep_shape v;
			ok = static_cast<bool>(in >> axis >> X >> Y >> Z >> S >> st >> alg >> v.chunk >> v.lines >> v.workgroups);
			if (ok)
				g_sweep_cache[shape_key { axis, X, Y, Z, S, st, alg, v.filter() }] = v;
		}
		else if (kind == "gradient" || kind == "gradient_field")
		{
			int X, Y, Z, S, st, alg, groups, stacked, order = 0;
			ok = static_cast<bool>(in >> X >> Y >> Z >> S >> st >> alg >> groups >> stacked);
			if (ok && !(in >> order)) // files written before the order field hold 8 numbers
				order = 0;
			ok = ok && (order == 0 || order == 1);
			if (ok)
				(kind == "gradient" ? g_tile_gradients : g_gradient_cache)[shape_key { -1, X, Y, Z, S, st, alg, false }] =
					gradient_shape { groups, stacked != 0, order };
		}
		else if (kind == "batch")
		{
			std::string key;
			std::array<int, 18> fields {};
			ok = static_cast<bool>(in >> key);
			for (int i = 0; i < 18 && ok; i++)
				ok = static_cast<bool>(in >> fields[i]);
			ok = ok && (fields[14] == 4 || fields[14] == 8);
			if (ok)
				g_batch_lines[key] = fields;
		}
		if (!ok)
			throw std::invalid_argument(std::string(path) + ":" + std::to_string(lineno) + ": not a tuning entry");
	}
}

// The automatic shape of an axis applied; false where it does not fit (a shape that the caller asked for may)
static bool apply_automatic(bfvm_ctx* ctx, int axis)
{
	try
	{
		apply_sweep_shape(ctx, axis, sweep_shape {});
		return true;
	}
	catch (const std::runtime_error&)
	{
		return false;
	}
}

static void autotune_axis(bfvm_ctx* ctx, int axis, int reps)
{
	const bool automatic =
		(ctx->chunk_request[axis] == 0 && ctx->lines_request[axis] == 0) || apply_automatic(ctx, axis);
	const bool filter = automatic && ctx->axes[axis].filter.blocks > 0;
	const shape_key key = key_of(ctx, axis, filter);
	sweep_shape shape;
	bool cached = false;
	{
		std::lock_guard<std::mutex> lock(g_cache_mutex);
		auto it = g_sweep_cache.find(key);
		if (it != g_sweep_cache.end())
		{
			shape = it->second;
			cached = true;
		}
	}
	if (!cached)
		shape = search_sweep(ctx, axis, filter, reps);
	apply_sweep_shape(ctx, axis, shape);
	if (!cached)
	{
		std::lock_guard<std::mutex> lock(g_cache_mutex);
		g_sweep_cache[key] = shape;
	}
}

void autotune_context(bfvm_ctx* ctx, bool tune_gradient)
{
	const int reps = 3;
	ctx->epoch++; // captured steps hold tables that are replaced below, also where tuning fails
	for (int axis = 0; axis < ctx->mesh.dims; axis++)
	{
		if (ctx->mesh.grid[axis] == 1 || ctx->algorithm != BFVM_SWEEP_PARTITIONED)
			continue;
		const sweep_shape asked { ctx->chunk_request[axis], ctx->lines_request[axis], ctx->sweep_workgroups[axis] };
		try
		{
			autotune_axis(ctx, axis, reps);
		}
		catch (...)
		{
			apply_sweep_shape(ctx, axis, asked);
			throw;
		}
	}
	if (tune_gradient && ctx->mesh.dims == 3)
	{
		const shape_key key = key_of(ctx, -1, false);
		gradient_shape best;
		bool cached = false;
		{
			std::lock_guard<std::mutex> lock(g_cache_mutex);
			auto it = g_gradient_cache.find(key);
			if (it != g_gradient_cache.end())
			{
				best = it->second;
				cached = true;
			}
		}
		if (!cached)
		{
			float best_t = 1e30f;
			auto consider = [&](const gradient_shape& shape) {
				ctx->gradient_groups = shape.groups;
				ctx->gradient_stacked = shape.stacked;
				ctx->gradient_order = shape.order;
				const float t = best_ms(ctx->stream, reps, [&] { launch_gradient(ctx); });
				if (t < best_t * 0.99f)
				{
					best_t = t;
					best = shape;
				}
			};
			consider(gradient_shape {}); // the automatic shape
			for (int order : { 0, 1 })
				for (bool stacked : { false, true })
					for (int g : { 4096, 8192, 16384, 32768, 65536 })
						consider(gradient_shape { g, stacked, order });
			std::lock_guard<std::mutex> lock(g_cache_mutex);
			g_gradient_cache[key] = best;
		}
		ctx->gradient_groups = best.groups;
		ctx->gradient_stacked = best.stacked;
		ctx->gradient_order = best.order;
	}
	BFVM_HIP(hipStreamSynchronize(ctx->stream));
}

} // namespace bfvm
