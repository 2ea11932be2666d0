#pragma once
struct __half;
