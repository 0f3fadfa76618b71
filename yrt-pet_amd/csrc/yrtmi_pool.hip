#include "yrtmi_pool.hpp"

#include <list>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace yrtmi
{

namespace
{

struct Block
{
	void* p;
	size_t bytes;
};

struct Device
{
	int contexts = 0;
	size_t kept = 0;
	std::list<Block> blocks;  // longest unused first
	std::vector<void*> unfreed;  // hipFree refused them: tried again
};

struct Pool
{
	std::mutex m;
	std::map<int, Device> dev;
	std::unordered_map<void*, size_t> live;
};

// never destroyed: handles may be dropped while the process ends
Pool& pool()
{
	static Pool* p = new Pool();
	return *p;
}

size_t rounded(size_t b)
{
	const size_t g = b < (size_t(1) << 20) ? 4096 : size_t(1) << 21;
	return (b + g - 1) / g * g;
}

// Gives v back to the driver.  Where that is refused (a thread is recording a
// graph) the memory is kept for a later try, and no error is left behind for
// the next call to find.
void freeAll(int device, const std::vector<void*>& v)
{
	for (void* p : v)
		if (hipFree(p) != hipSuccess)
		{
			(void)hipGetLastError();
			Pool& P = pool();
			std::lock_guard<std::mutex> lk(P.m);
			P.dev[device].unfreed.push_back(p);
		}
}

// under the mutex
void takeAll(Device& d, std::vector<void*>& out)
{
	for (const Block& b : d.blocks)
		out.push_back(b.p);
	out.insert(out.end(), d.unfreed.begin(), d.unfreed.end());
	d.blocks.clear();
	d.unfreed.clear();
	d.kept = 0;
}

}  // namespace

void poolRetain(int device)
{
	Pool& P = pool();
	std::lock_guard<std::mutex> lk(P.m);
	P.dev[device].contexts++;
}

void poolRelease(int device)
{
	Pool& P = pool();
	std::vector<void*> drop;
	{
		std::lock_guard<std::mutex> lk(P.m);
		Device& d = P.dev[device];
		if (--d.contexts <= 0)
			takeAll(d, drop);
	}
	freeAll(device, drop);
}

void poolTrim(int device)
{
	Pool& P = pool();
	std::vector<void*> drop;
	{
		std::lock_guard<std::mutex> lk(P.m);
		takeAll(P.dev[device], drop);
	}
	freeAll(device, drop);
}

size_t poolKept(int device)
{
	Pool& P = pool();
	std::lock_guard<std::mutex> lk(P.m);
	return P.dev[device].kept;
}

hipError_t poolMalloc(int device, void** out, size_t bytes)
{
	hipError_t e = hipMalloc(out, bytes);
	if (e != hipSuccess)
	{
		(void)hipGetLastError();
		poolTrim(device);
		e = hipMalloc(out, bytes);
	}
	return e;
}

hipError_t poolAlloc(int device, void** out, size_t bytes, bool exact)
{
	Pool& P = pool();
	const size_t need = rounded(bytes), slack = exact ? 0 : need / 4 + (size_t(1) << 20);
	{
		std::lock_guard<std::mutex> lk(P.m);
		Device& d = P.dev[device];
		auto best = d.blocks.end();
		for (auto it = d.blocks.begin(); it != d.blocks.end(); ++it)
			if (it->bytes >= need && it->bytes <= need + slack &&
			    (best == d.blocks.end() || it->bytes < best->bytes))
				best = it;
		if (best != d.blocks.end())
		{
			*out = best->p;
			P.live[best->p] = best->bytes;
			d.kept -= best->bytes;
			d.blocks.erase(best);
			return hipSuccess;
		}
	}
	void* p = nullptr;
	const hipError_t e = poolMalloc(device, &p, need);
	if (e != hipSuccess)
	{
		*out = nullptr;
		return e;
	}
	*out = p;
	std::lock_guard<std::mutex> lk(P.m);
	P.live[p] = need;
	return hipSuccess;
}

void poolFree(int device, void* p, bool idle)
{
	if (p == nullptr)
		return;
	Pool& P = pool();
	std::vector<void*> drop;
	{
		std::lock_guard<std::mutex> lk(P.m);
		Device& d = P.dev[device];
		const auto it = P.live.find(p);
		const size_t bytes = it != P.live.end() ? it->second : 0;
		if (it != P.live.end())
			P.live.erase(it);
		if (!idle || d.contexts <= 0 || bytes == 0 || bytes > kPoolBytes)
			drop.push_back(p);
		else
		{
			d.blocks.push_back({p, bytes});
			d.kept += bytes;
			while (d.kept > kPoolBytes)
			{
				drop.push_back(d.blocks.front().p);
				d.kept -= d.blocks.front().bytes;
				d.blocks.pop_front();
			}
		}
	}
	freeAll(device, drop);
}

bool poolQuiesce(int device)
{
	int cur = device;
	(void)hipGetDevice(&cur);
	(void)hipSetDevice(device);
	const hipError_t e = hipDeviceSynchronize();
	if (e != hipSuccess)
		(void)hipGetLastError();
	(void)hipSetDevice(cur);
	return e == hipSuccess;
}

}  // namespace yrtmi
