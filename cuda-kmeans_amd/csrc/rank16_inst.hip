/* One instantiation of the half-precision ranking sweep and its exact pass: KMX_KB blocks of 16 dimensions per row (given on the command line). */
#include "rank16_exact_impl.h"

#ifndef KMX_KB
#error "compile with -DKMX_KB=<blocks of 16 dimensions per row>"
#endif

#define KMX_CAT2(a, b) a##b
#define KMX_CAT(a, b) KMX_CAT2(a, b)

namespace kmx {

int KMX_CAT(launch_rank16_, KMX_KB)(const AssignArgs& a, const Rank16Args& w, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev)
{
	return launch_rank16_kb<KMX_KB>(a, w, exec, ws, dev);
}

int KMX_CAT(launch_listed_exact_, KMX_KB)(const AssignArgs& a, const ExactArgs<float>& w, const DeviceInfo& dev)
{
	return launch_listed_exact_kb<KMX_KB, float>(a, w, dev);
}

int KMX_CAT(launch_listed_exact_, KMX_KB)(const AssignArgs& a, const ExactArgs<double>& w, const DeviceInfo& dev)
{
	return launch_listed_exact_kb<KMX_KB, double>(a, w, dev);
}

} // namespace kmx
