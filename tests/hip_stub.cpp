// A stand-in for the HIP runtime on a machine without a GPU: device memory is
// host memory, nothing runs, and every kernel launch is recorded with its name,
// grid and arguments. Loaded with RTLD_GLOBAL before libnnc_hip.so, whose calls
// then resolve to it, so a test can check on the CPU what the host code
// launches, on which allocations, and which of those live on.
#include "../libllmcpu_amd/csrc/kernels.h"

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace
{
	struct launch
	{
		std::string name;
		dim3 grid;
		nnchip::gemv_params gemv; // kernels that take them
		nnchip::decode_params attn;
		const char* split; // tiled3 kernels: the operands
		bool captured;
	};
	std::map<const char*, size_t> g_live; // device allocations
	std::map<const void*, std::string> g_names; // host function -> kernel
	std::vector<launch> g_launches;
	bool g_capturing = false, g_invalid = false; // a capture that met a call it does not allow
	struct
	{
		dim3 grid, block;
		size_t lds;
		hipStream_t stream;
	} g_config;
	char g_symbol[NNC_STUB_SYMBOL_BYTES];

	hipError_t unsafe()
	{
		if (g_capturing) g_invalid = true;
		return g_capturing ? hipErrorStreamCaptureUnsupported : hipSuccess;
	}
}

extern "C" {

// ---- what a test asks ----
void stub_capture(int on)
{
	g_capturing = on != 0;
	if (on) g_invalid = false;
}
int stub_capture_invalid() { return g_invalid; }
int stub_launches() { return static_cast<int>(g_launches.size()); }
void stub_clear() { g_launches.clear(); }
const char* stub_name(int i) { return g_launches[i].name.c_str(); }
int stub_captured(int i) { return g_launches[i].captured; }
// The staged X (0), a gemv's partial sums (1), the tiled3 operands (2) or the
// attention partials (3) of launch i, null where it has none.
const void* stub_pointer(int i, int what)
{
	const launch& l = g_launches[i];
	if (what == 0) return l.gemv.xs;
	if (what == 1) return l.gemv.n_split > 1 ? l.gemv.part : nullptr;
	if (what == 2) return l.split;
	return l.attn.n_split > 1 ? l.attn.part : nullptr;
}
// n_batch, cols, rows, x_tiles, n_split of a gemv launch.
void stub_gemv(int i, int* out)
{
	const nnchip::gemv_params& p = g_launches[i].gemv;
	const int v[5] = {p.n_batch, p.cols, p.rows, p.x_tiles, p.n_split};
	std::memcpy(out, v, sizeof v);
}
// Bytes from p to the end of its allocation, 0 when it is freed.
size_t stub_bytes_left(const void* p)
{
	const char* c = static_cast<const char*>(p);
	auto it = g_live.upper_bound(c);
	if (it == g_live.begin()) return 0;
	--it;
	return c < it->first + it->second ? static_cast<size_t>(it->first + it->second - c) : 0;
}
size_t stub_live_bytes()
{
	size_t n = 0;
	for (const auto& a : g_live) n += a.second;
	return n;
}

// ---- the runtime ----
hipError_t hipMalloc(void** p, size_t n)
{
	if (hipError_t e = unsafe()) return e;
	*p = std::malloc(n ? n : 1);
	g_live[static_cast<char*>(*p)] = n;
	return hipSuccess;
}
hipError_t hipFree(void* p)
{
	if (hipError_t e = unsafe()) return e;
	if (p && !g_live.erase(static_cast<char*>(p))) return hipErrorInvalidValue;
	// (not given back to malloc, so that an address names one allocation)
	return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
	*p = std::malloc(n);
	return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
	std::free(p);
	return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
	*s = reinterpret_cast<hipStream_t>(&g_config);
	return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return unsafe(); }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st)
{
	*st = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
	return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
	*e = reinterpret_cast<hipEvent_t>(&g_config);
	return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return unsafe(); }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n)
{
	*n = 1;
	return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
	*d = 0;
	return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int)
{
	*v = 256; // compute units
	return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600*, int) { return hipErrorNotSupported; }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
	*p = g_symbol;
	return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }

void** __hipRegisterFatBinary(const void*)
{
	static void* modules;
	return &modules;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
	g_names[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
	g_config = {grid, block, lds, stream};
	return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
	*grid = g_config.grid;
	*block = g_config.block;
	*lds = g_config.lds;
	*stream = g_config.stream;
	return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3, void** args, size_t, hipStream_t)
{
	launch l{};
	l.name = g_names[fn];
	l.grid = grid;
	l.captured = g_capturing;
	if (l.name.find("gemv_params") != std::string::npos) l.gemv = *static_cast<nnchip::gemv_params*>(args[0]);
	if (l.name.find("decode_params") != std::string::npos) l.attn = *static_cast<nnchip::decode_params*>(args[0]);
	if (l.name.find("tiled3") != std::string::npos) l.split = *static_cast<const char**>(args[1]);
	g_launches.push_back(l);
	return hipSuccess;
}
}
