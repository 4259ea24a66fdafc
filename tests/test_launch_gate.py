"""The gate between threads that launch calls which had been put aside and a thread that gives device memory back (launch_gate.h), compiled
by itself for the CPU."""
import os
import subprocess

import neoml_amd

PROGRAM = r"""
#include "launch_gate.h"
#include <chrono>
#include <cstdio>

static nh::CLaunchGate gate;

struct CWaiter {
	std::atomic<bool> Done{ false };
	std::thread Thread{ [this]() { gate.WaitForThoseInside(); Done = true; } };
	~CWaiter() { Thread.join(); }
	// whether it has returned, given time
	bool Returns( int milliseconds )
	{
		for( int i = 0; i < milliseconds && !Done; ++i ) {
			std::this_thread::sleep_for( std::chrono::milliseconds( 1 ) );
		}
		return Done;
	}
};

// a thread that goes in and out when it is told to
struct CLauncher {
	std::atomic<int> Want{ 0 }, Is{ 0 };
	std::thread Thread{ [this]() {
		nh::CLaunchGate::CThread place( gate );
		while( Want >= 0 ) {
			if( Want != Is ) {
				Want != 0 ? place.Enter() : place.Leave();
				Is = Want != 0 ? 1 : 0;
			}
			std::this_thread::yield();
		}
		if( Is != 0 ) {
			place.Leave();
		}
	} };
	void Set( int inside )
	{
		Want = inside;
		while( Is != inside ) {
			std::this_thread::yield();
		}
	}
	~CLauncher() { Want = -1; Thread.join(); }
};

#define CHECK( what ) if( !( what ) ) { std::printf( "failed: %s\n", #what ); std::fflush( stdout ); std::_Exit( 1 ); }

int main()
{
	{
		CWaiter none;
		CHECK( none.Returns( 5000 ) );
	}
	{
		CLauncher first, second;
		first.Set( 1 );
		CWaiter waiter;
		CHECK( !waiter.Returns( 100 ) );
		// who goes in beside one who waits neither waits nor is waited for
		second.Set( 1 );
		CWaiter later;
		CHECK( !waiter.Returns( 50 ) );
		first.Set( 0 );
		CHECK( waiter.Returns( 5000 ) );
		CHECK( !later.Returns( 50 ) );
		first.Set( 1 );
		second.Set( 0 );
		CHECK( later.Returns( 5000 ) );
		// inside again is not inside still
		CWaiter again;
		CHECK( !again.Returns( 50 ) );
		first.Set( 0 );
		first.Set( 1 );
		CHECK( again.Returns( 5000 ) );
	}
	{
		CWaiter ended;
		CHECK( ended.Returns( 5000 ) );
	}
	std::printf( "ok\n" );
	return 0;
}
"""


def test_waits_for_those_inside_only(tmp_path):
    source, program = str(tmp_path / "gate.cpp"), str(tmp_path / "gate")
    with open(source, "w") as f:
        f.write(PROGRAM)
    include = os.path.join(os.path.dirname(neoml_amd.__file__), "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I", include, source, "-o", program], check=True)
    ran = subprocess.run([program], stdout=subprocess.PIPE, text=True, timeout=60)
    assert ran.returncode == 0 and ran.stdout == "ok\n", ran.stdout
